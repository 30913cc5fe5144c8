// int4 x int4 GEMM on the FP6 matrix path straight from packed nibbles, exact: outputs that fill the compute units with tiles of
// 128, 192 or 256 rows x 256 columns.
//
// An FP6 E2M3 number with the bits 0mmmmm... below is the plain binary integer / 8: the magnitudes 0 .. 15 of 1/8 have the codes
// 000000 .. 001111 (0 .. 7 are its subnormals, 8 .. 15 the numbers from 1).  So u = code + 8 in 0 .. 15, a nibble with its top bit
// flipped, IS an E2M3 operand once the nibbles of a word stand six bits apart with two zero bits between them, and
//   sum a b = sum ua ub - 8 sum ua - 8 sum ub + 64 K.
// v_mfma_f32_32x32x64_f8f6f4 takes 64 k in the 32 cycles that v_mfma_i32_32x32x32_i8 takes for 32.  Every product is an
// integer / 64 of at most 225, every partial sum an integer / 64 below 2^24 (kSegment below), so the result is the integer dot product.
//
// What it does without: converting signs (the sum of a row's codes costs less, see `ones`), and a second copy of either operand (the
// format of gemm_f6.hip, 6 bits in memory, moves 1.5 times the bytes through L2 and LDS).
#include "qr_e2m3.h"
#include "qr_epilogue.h"

namespace {

typedef int i32x6 __attribute__((ext_vector_type(6)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

// Stages (of 256 k) between two corrections of the accumulators by the row sums.  Between them a sum is at most 225 per k over 192 stages
// on top of the corrected sum of everything before, 64 per k: (225 * 192 + 64 * (512 - 192)) * 256 = 16.3e6 < 2^24 for K up to 131072.
constexpr int kSegment = 192;

// LDS bytes: stage buffers, then scales ([256] sB, [256] bias, [BM] sA in fp16; KG = 1: of two tiles), row sums of both operands, and
// (KG = 1, whose stage buffers hold the next tile's first stages by then) the output slabs
constexpr int e2m3_lds(int BM, int KG) {
    return KG == 1 ? 2 * (BM + 256) * 128 + 2 * (512 + BM) * 2 + (BM + 256) * 4 + 16384
                   : 3 * (BM + 256) * 128 + (512 + BM) * 2 + 2 * (BM + 256) * 4;
}
// Four waves, ONE per SIMD, each with a wave tile of 128 (96) x 128: 16 (12) accumulator tiles, up to all 256 accumulation registers.
//   KG = 1   waves 2 (M) x 2 (N), BM = 256 or 192, whole K per wave
//   KG = 2   waves 2 (N) x 2 (K), BM = 128: the K-groups take alternate pairs of sub-steps and exchange half their accumulators at the end
//
// A stage is 256 k (a 128-byte line per row), loaded straight into LDS (buffer_load ... lds; the XOR-keyed layout is made by permuting
// which 16 bytes of a line a lane fetches), and a sub-step is 64 k: 16 bytes per lane and fragment of 32 rows.  A wave hides everything
// under its own matrix instructions, in explicit slots: one matrix instruction and an even share of the 14 vector instructions per
// fragment that spread the NEXT sub-step's nibbles; behind a fragment's last one the read of the sub-step AFTER that into the same
// registers; loads of the stage after next, one in two (KG = 2: three) slots (one in every slot, they back up behind one another: 59
// instead of 55 cycles per slot).  A scheduling barrier after every slot keeps this order.
//
// KG = 1: a workgroup takes `count` tiles, place(0), place(1) .., without a gap in this pipeline: where the loop over a tile's K would
// load stages past its end, it loads the next tile's first ones, and the next tile's first sub-step is spread before the epilogue.
// With a workgroup per tile every tile paid some 2-3 us for launch, first loads and first sub-step: 32768 x 4096 x 1024 138 -> 122 us,
// 32768 x 11008 x 4096 835 -> 812, 32768 x 4096 x 11008 710 -> 690.  (The turn is prepared between two runs of the stage loop: a branch
// for it inside the loop, or one that lets the epilogue's stores pass the first barrier, costs 6 % of every stage.)
//
// What bounds it (256 rows, 32768 x 4096 x 11008): a wave issues an instruction in about 5 cycles, and a sub-step has 20 matrix and 112
// vector instructions, 8 LDS reads, 4 loads and some 20 others.  Counters: 61 cycles of 1.9 GHz per accumulator tile and sub-step over the
// whole launch, 57 without the 6 us behind the loop of every tile (3 us of arithmetic with one wave per SIMD, then the compute units write
// 33 MB at a time), where the matrix unit alone would need 36: it is busy for 0.60 of the launch, the vector unit for 0.52.  The clock is
// the power limit's (2.4 GHz without load; 2.2 at K = 4096, where the matrix unit is busy for 0.51).  The whole launch is 4.15-4.3e15
// operations per second, 7.1e15 being what the matrix instruction sustains on these operands with nothing else going on (the int8 one
// 3.9-4.2e15): 690-712 us against 870-890 of the int8 kernel with the same tiles; 32768 x 11008 x 4096 812 us (1010; 850 with a branch around
// every store), 8192 x 5120 x 5120 124 (146), 1777 x 8192 x 28672 195 (244), 2048 x 4096 x 11008 53-54 (58-66).  Delaying the first workgroups by 0 .. 8 us, so
// that compute units do not write at once, changed nothing.
template <bool DEQ, bool RAGGED, int BM, int KG, class Place>
__device__ __forceinline__ void e2m3_tiles(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int count, Place place) {
    static_assert(KG == 1 ? (BM == 256 || BM == 192) : BM == 128, "wave tiles of 128 x 128 or 96 x 128");
    constexpr int NT = 256;
    constexpr int TM = KG == 1 ? BM / 2 : BM, IM = TM / 32, JN = 4;
    constexpr int STAGE = (BM + 256) * 128;                 // bytes of a stage buffer
    constexpr int NL = STAGE / 16 / NT;                     // loads per thread and stage
    constexpr int NF = IM + JN;                             // fragments of a sub-step
    constexpr int NBUF = KG == 1 ? 2 : 3;
    constexpr int SU = 4 / KG;                              // sub-steps of a stage that a wave takes
    constexpr int SUM_B = KG == 1 ? 2 : 4;                  // fragments of B whose rows a wave adds up (KG = 1: the other two are the other wave row's)
    constexpr int NS = 2 + SUM_B;                           // fragments whose rows a wave adds up
    constexpr int NU = IM * JN + NS;                        // matrix instructions (= slots) of a sub-step
    constexpr int UNP = 14 * NF;                            // vector instructions that spread a sub-step's fragments
    extern __shared__ u32x4 e2m3_smem[];
    char* const lds = (char*)e2m3_smem;
    f16* scales = (f16*)(lds + NBUF * STAGE);               // (of the tile at hand)
    float* const rowsum = (float*)(scales + (KG == 1 ? 2 : 1) * (512 + BM));     // [KG][BM] of A
    float* const colsum = rowsum + KG * BM;                 // [KG][256] of B

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = KG == 1 ? wave >> 1 : 0, wn = wave & 1, kg = KG == 1 ? 0 : wave >> 1;
    const int khalf = lane >> 5;
    const int stages = (Kb + 127) / 128;
    auto slot8 = [](int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); };

    // loads: chunk tid + i * 256 of a stage is 16 bytes of row tid / 8 + 32 i, at LDS position (row, tid % 8): the lane fetches the piece
    // that the layout keeps there (the key is the same for all of a lane's rows)
    const int srow = tid >> 3, piece = ((tid & 7) ^ ((srow >> 1) & 7)) * 16;
    Origin at = place(0);
    u32 goff[NL];
    auto aim = [&](Origin o) {
        int row0 = srow;
        asm volatile("" : "+v"(row0));                      // (computed here, not kept over the tiles: registers are full)
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int row = row0 + i * 32;
            int gr = row < BM ? o.m0 + row : o.n0 + row - BM;
            const int lim = row < BM ? M - 1 : N - 1;
            gr = gr < lim ? gr : lim;
            goff[i] = (u32)gr * (u32)Kb + (u32)piece;
        }
    };
    aim(at);
    bool more = false;                                      // stages past the end are the next tile's
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)((u32)M * (u32)Kb), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)((u32)N * (u32)Kb), 0x00020000);
    // (where there is no next tile, stages past the end repeat the last one into a buffer that nobody reads: every stage issues the
    // same number of loads)
    auto load1 = [&](int st, int buf, int i) __attribute__((always_inline)) {
        const int kb = (st < stages ? st : more ? st - stages : stages - 1) * 128;
        __attribute__((address_space(3))) void* dst =
            (__attribute__((address_space(3))) void*)(lds + buf * STAGE + (i * NT + wave * 64) * 16);
        // pieces past the end of a row are sent beyond the buffer's range and arrive as zeros: codes 0 (an operand is a multiple of 32
        // bytes below 4 GiB: at most 0xFFFFFFE0)
        const u32 off = RAGGED && kb + piece >= Kb ? 0xFFFFFFE0u : goff[i];
        if (i * 32 < BM) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, dst, 16, off, kb, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, dst, 16, off, kb, 0, 0);
    };

    f32x16 acc[IM][JN];

    // Group of 32 rows that fragment i of A / j of B holds.  Waves that share rows of an operand hold its fragments in different orders, so that
    // fragments 0 and 1, whose rows a wave adds up, are different rows in each; K-group 1 holds the halves of B swapped, so that
    // either group keeps accumulator columns j = 0, 1 and sends 2, 3.
    auto ga = [&](int i) { return IM == 4 ? i ^ (2 * wn) : (wn ? 2 - i : i); };
    auto gb = [&](int j) { return KG == 1 ? j ^ (2 * wm) : j ^ (2 * kg); };
    // byte addresses of the fragments of sub-step u: one base per pair of fragments that keep their distance (ga, gb move pairs)
    constexpr int NA = IM == 4 ? 2 : 3, NB = NA + 2;
    auto base_of = [](int f) { return f < IM ? (IM == 4 ? f >> 1 : f) : NA + ((f - IM) >> 1); };
    auto dist_of = [](int f) { return f < IM ? (IM == 4 ? (f & 1) * 4096 : 0) : ((f - IM) & 1) * 4096; };
    int base[SU][NB];
#pragma unroll
    for (int u = 0; u < SU; ++u) {
        const int chunk = 2 * (KG == 1 ? u : 2 * kg + u) + khalf;
#pragma unroll
        for (int f = 0; f < NF; ++f)
            if (dist_of(f) == 0)
                base[u][base_of(f)] = 16 * (f < IM ? slot8(wm * TM + ga(f) * 32 + (lane & 31), chunk)
                                                   : slot8(BM + wn * 128 + gb(f - IM) * 32 + (lane & 31), chunk));
    }
    struct Packed {
        u32x4 f[NF];
    };
    struct Ops {
        u32 d[NF][6];
    };
    auto read1 = [&](int u, int f, int buf_off, Packed& p) __attribute__((always_inline)) {
        p.f[f] = *(const u32x4*)(lds + (base[u][base_of(f)] + buf_off) + dist_of(f));
    };

    // Spreading (qr_e2m3.h), seven instructions per two words: y rotated by 2, then for each word (x & mask) ^ top bits of its eight nibbles' places, then
    // ^ (rotated y & mask), one v_bitop3_b32 each (one operand may be scalar: the masks of x are held in vector registers).
    u32 x0, x1, x2, y0, y1, y2, c0, c1, c2;
    asm("v_mov_b32 %0, %1" : "=v"(x0) : "n"(kSpreadX[0]));
    asm("v_mov_b32 %0, %1" : "=v"(x1) : "n"(kSpreadX[1]));
    asm("v_mov_b32 %0, %1" : "=v"(x2) : "n"(kSpreadX[2]));
    asm("s_mov_b32 %0, %1" : "=s"(y0) : "n"(kSpreadY[0]));
    asm("s_mov_b32 %0, %1" : "=s"(y1) : "n"(kSpreadY[1]));
    asm("s_mov_b32 %0, %1" : "=s"(y2) : "n"(kSpreadY[2]));
    asm("s_mov_b32 %0, %1" : "=s"(c0) : "n"(kSpreadFlip[0]));
    asm("s_mov_b32 %0, %1" : "=s"(c1) : "n"(kSpreadFlip[1]));
    asm("s_mov_b32 %0, %1" : "=s"(c2) : "n"(kSpreadFlip[2]));
    // the order in which a sub-step's fragments are spread (and read again)
    constexpr int order4[8] = {0, 2, 1, 3, 4, 6, 5, 7}, order3[7] = {0, 2, 1, 3, 5, 4, 6};
    auto frag_at = [&](int t) { return IM == 4 ? order4[t] : order3[t]; };
    // instruction n of UNP
    auto spread1 = [&](Packed& p, Ops& o, int n) __attribute__((always_inline)) {
        constexpr u32 AND_XOR = 0x6a;                       // (a & b) ^ c
        const int t = n / 7, kind = n % 7, f = frag_at(t >> 1), h = t & 1;
        u32* d = &o.d[f][3 * h];
        const u32 x = p.f[f][2 * h], y = p.f[f][2 * h + 1];
        if (kind == 0) p.f[f][2 * h + 1] = __builtin_amdgcn_alignbit(y, y, 30);
        else if (kind == 1) d[0] = __builtin_amdgcn_bitop3_b32(x, x0, c0, AND_XOR);
        else if (kind == 2) d[1] = __builtin_amdgcn_bitop3_b32(x, x1, c1, AND_XOR);
        else if (kind == 3) d[2] = __builtin_amdgcn_bitop3_b32(x, x2, c2, AND_XOR);
        else if (kind == 4) d[0] = __builtin_amdgcn_bitop3_b32(y, y0, d[0], AND_XOR);
        else if (kind == 5) d[1] = __builtin_amdgcn_bitop3_b32(y, y1, d[1], AND_XOR);
        else d[2] = __builtin_amdgcn_bitop3_b32(y, y2, d[2], AND_XOR);
    };
    // (formats: 2 = FP6 E2M3, 4 = FP4 E2M1; no scales)
    auto opnd = [&](const Ops& o, int f) {
        return i32x8{(int)o.d[f][0], (int)o.d[f][1], (int)o.d[f][2], (int)o.d[f][3], (int)o.d[f][4], (int)o.d[f][5], 0, 0};
    };
    auto mfma1 = [&](const Ops& o, int q) __attribute__((always_inline)) {
        const int i = q / JN, j = q % JN;
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(opnd(o, IM + j), opnd(o, i), acc[i][j], 2, 2, 0, 0, 0, 0);
    };
    // Sums of rows: 16 x 16 x 128 instructions, half the time of the others, in which a fragment's 64 lanes count as 16 rows x four groups of 32 k.
    // The first operand has ones (FP4) in row 2 t for lanes with rows 0 .. 15 of summed fragment t, in row 2 t + 1 for those with rows
    // 16 .. 31, and zeros elsewhere, so that all fragments share one accumulator: lanes 16 g .. 16 g + 15 end with the sums of fragments
    // 2 g (registers 0, 1) and 2 g + 1 (registers 2, 3).  (Dot products of the packed words, v_dot8_i32_i4, stall the wave behind the matrix
    // instructions: 14 cycles each, 16-24 per sub-step.  The accumulator is spelled out as vector registers: the accumulation
    // registers are full, and the compiler would move tiles out of them and back.)
    auto summed = [](int t) { return t < 2 ? t : IM + t - 2; };
    i32x4 ones[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        int v = (lane & 15) == 2 * t + ((lane >> 4) & 1) ? 0x22222222 : 0;
        asm("" : "+v"(v));
        ones[t] = i32x4{v, v, v, v};
    }
    f32x4 sums = {0.f, 0.f, 0.f, 0.f};
    auto sum1 = [&](const Ops& o, int t) __attribute__((always_inline)) {
        const int f = summed(t);
        const i32x6 u = {(int)o.d[f][0], (int)o.d[f][1], (int)o.d[f][2], (int)o.d[f][3], (int)o.d[f][4], (int)o.d[f][5]};
        asm("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:4 blgp:2" : "+v"(sums) : "v"(ones[t]), "v"(u));
    };

    // One sub-step: multiply `cur`, spread `p` into `nxt`, read sub-step RU of the stage buffer at buf_off into `p` behind it, and load chunks
    // LOAD0 .. LOAD1 of stage load_st into buffer load_buf from slot LSLOT on. 
    // BSLOT >= 0: the stage's barrier stands in this slot (at most ALLOWED of the wave's memory operations still in flight), and no read is
    // issued before it.
    constexpr int EVERY = KG == 1 ? 2 : 3;                  // slots from one load to the next
#define QR_E2M3_BARRIER(ALLOWED) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(ALLOWED) : "memory");
    auto substep = [&](const Ops& cur, Ops& nxt, Packed& p, auto ru, int buf_off, auto bslot, auto allowed, int load_st, int load_buf,
                       auto load0, auto load1_, auto lslot) __attribute__((always_inline)) {
        constexpr int RU = decltype(ru)::value, BSLOT = decltype(bslot)::value, ALLOWED = decltype(allowed)::value;
        constexpr int LOAD0 = decltype(load0)::value, LOAD1 = decltype(load1_)::value, LSLOT = decltype(lslot)::value;
        static_assert(LOAD1 <= LOAD0 || LOAD1 - LOAD0 <= (NU - LSLOT + EVERY - 1) / EVERY, "every load has a slot");
        static_for<NU>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value, done_sums = q * NS / NU;
            if constexpr ((q + 1) * NS / NU > done_sums) sum1(cur, done_sums);
            else mfma1(cur, q - done_sums);
            constexpr int N0 = q * UNP / NU, N1 = (q + 1) * UNP / NU;
            static_for<N1 - N0>([&](auto nc) __attribute__((always_inline)) { spread1(p, nxt, N0 + decltype(nc)::value); });
            if constexpr (q == BSLOT) QR_E2M3_BARRIER(ALLOWED)
            static_for<NF>([&](auto tc) __attribute__((always_inline)) {
                constexpr int t = decltype(tc)::value;
                constexpr int done = ((t + 1) * 14 * NU + UNP - 1) / UNP - 1;    // slot of the fragment's last instruction
                if constexpr (q == (done < BSLOT ? BSLOT : done)) read1(RU, frag_at(t), buf_off, p);
            });
            if constexpr (LOAD1 > LOAD0 && q >= LSLOT && (q - LSLOT) % EVERY == 0 && LOAD0 + (q - LSLOT) / EVERY < LOAD1)
                load1(load_st, load_buf, LOAD0 + (q - LSLOT) / EVERY);
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // The epilogue's scales and bias are fetched first and parked in LDS: a load in the epilogue would wait for the stores before it.
    // (Indices clamped to the matrix: what belongs to rows and columns beyond it is never stored.)
    f16 pre_sb = (f16)0, pre_bi = (f16)-0.0f, pre_sa = (f16)0;
    auto fetch_scales = [&](Origin o) {
        if (!DEQ) return;
        const int col = o.n0 + tid < N ? o.n0 + tid : N - 1, row = o.m0 + tid < M ? o.m0 + tid : M - 1;
        pre_sb = sB[col], pre_sa = sA[row];
        if (bias) pre_bi = bias[col];
    };
    auto park_scales = [&] {
        if (!DEQ) return;
        scales[tid] = pre_sb;
        scales[256 + tid] = pre_bi;
        if (tid < BM) scales[512 + tid] = pre_sa;
    };
    fetch_scales(at);
    // Loads of a stage: KG = 1 in sub-steps 2 and 3 of the stage two before it (once its buffer is free), KG = 2 in the two sub-steps of the
    // stage three before it
    constexpr int L2 = (NU - 4 + EVERY - 1) / EVERY < NL ? (NU - 4 + EVERY - 1) / EVERY : NL;
#pragma unroll
    for (int s = 0; s < NBUF; ++s)
#pragma unroll
        for (int i = 0; i < NL; ++i) load1(s, s, i);
    QR_E2M3_BARRIER((NBUF - 1) * NL)
    park_scales();
    Packed pk;
    Ops ops[2];
#pragma unroll
    for (int f = 0; f < NF; ++f) read1(0, f, 0, pk);
    static_for<UNP>([&](auto nc) __attribute__((always_inline)) { spread1(pk, ops[0], decltype(nc)::value); });
#pragma unroll
    for (int t = 0; t < NF; ++t) read1(1, frag_at(t), 0, pk);   // in the order of the loop, whose waits count reads

    int off = 0, nxt = STAGE, buf = 0;                          // stage ks is in buffer `buf` at `off`, the next one at `nxt`
    for (int t = 0;;) {
    Origin then{0, 0};                                          // the tile after this one
    // (zeros by matrix instructions: one each, and no vector of zeros that has to live somewhere)
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
            f32x16 none;
#pragma unroll
            for (int v = 0; v < 16; ++v) none[v] = 0.f;
            float zero = 0.f;
            asm volatile("" : "+v"(zero));                      // (or the compiler makes one tile of zeros and copies it)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(zero, zero, none, 0, 0, 0);
        }
    for (int ks = 0, seg = 0; ks < stages;) {
        const int end = seg + kSegment < stages ? seg + kSegment : stages;      // the accumulators are corrected here
        if constexpr (KG == 1) {
            // Stage ks is read during sub-steps 2, 3 of stage ks - 1 and 0, 1 of stage ks.  The barrier early in sub-step 2: stage ks + 1 has
            // landed, everybody is done with stage ks.
            const int turn = stages - 2;                        // from this stage on the loads are the next tile's
            if (ks == turn && t + 1 < count) {
                then = place(t + 1);
                aim(then);
                fetch_scales(then);
                more = true;
            }
            const int stop = ks < turn && turn < end ? turn : end;
            for (; ks < stop; ++ks) {
                substep(ops[0], ops[1], pk, IC<2>(), off, IC<-1>(), IC<0>(), 0, 0, IC<0>(), IC<0>(), IC<0>());
                substep(ops[1], ops[0], pk, IC<3>(), off, IC<-1>(), IC<0>(), 0, 0, IC<0>(), IC<0>(), IC<0>());
                substep(ops[0], ops[1], pk, IC<0>(), nxt, IC<3>(), IC<0>(), ks + 2, buf, IC<0>(), IC<L2>(), IC<4>());
                substep(ops[1], ops[0], pk, IC<1>(), nxt, IC<-1>(), IC<0>(), ks + 2, buf, IC<L2>(), IC<NL>(), IC<0>());
                off = STAGE - off;
                nxt = STAGE - nxt;
                buf ^= 1;
            }
        } else {
            // Sub-step v of stage ks is read during sub-step v of stage ks - 1.  The barrier early in the first sub-step: stage ks + 1 has landed
            // (at most stage ks + 2 is out), everybody is done with stage ks.
            for (; ks < end; ++ks) {
                substep(ops[0], ops[1], pk, IC<0>(), nxt, IC<3>(), IC<NL>(), ks + 3, buf, IC<0>(), IC<L2>(), IC<4>());
                substep(ops[1], ops[0], pk, IC<1>(), nxt, IC<-1>(), IC<0>(), ks + 3, buf, IC<L2>(), IC<NL>(), IC<0>());
                nxt = nxt == 2 * STAGE ? 0 : nxt + STAGE;
                buf = buf == 2 ? 0 : buf + 1;
            }
        }
        if (ks < end) continue;
        // sum a b / 64 = acc - (sum of the row's u) / 8 - (sum of the column's u) / 8 + number of k: a matrix instruction with k = 2 per tile
        // (each K-group corrects its own part by its own sums).  The compiler does not see that `sums` comes from a matrix instruction: its
        // last result is waited for by hand.
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(sums)::"memory");
        int ls = lane;
        asm volatile("" : "+v"(ls));
        if (ls < 8 * NS) {
            const int g = ls >> 4, r = ls & 15;         // fragments 2 g, 2 g + 1: two of A, then those of B
            float* const s = g == 0 ? rowsum + kg * BM + wm * TM : colsum + kg * 256 + wn * 128;
            const int f0 = g == 0 ? ga(0) : g == 1 ? gb(0) : gb(2), f1 = g == 0 ? ga(1) : g == 1 ? gb(1) : gb(3);
            s[f0 * 32 + r] = sums[0];
            s[f0 * 32 + 16 + r] = sums[1];
            s[f1 * 32 + r] = sums[2];
            s[f1 * 32 + 16 + r] = sums[3];
        }
        __syncthreads();
        const float terms = (float)((end - seg) * (256 / KG));
#pragma unroll
        for (int i = 0; i < IM; ++i) {
            const float rs = terms - rowsum[kg * BM + wm * TM + ga(i) * 32 + (ls & 31)];
#pragma unroll
            for (int j = 0; j < JN; ++j) {
                const float cs = colsum[kg * 256 + wn * 128 + gb(j) * 32 + (ls & 31)];
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32((ls >> 5) ? 1.f : -cs, (ls >> 5) ? rs : 1.f, acc[i][j], 0, 0, 0);
            }
        }
        sums = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // (the sums are read before the next ones are written)
        seg = end;
    }
    // repeats of the last stage are still landing in the stage buffers, which the K-groups' exchange and the next user of this LDS take
    const bool last = t + 1 == count;
    if (KG == 2 || last) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (KG == 2) __syncthreads();
    if constexpr (KG == 2) {
        // the K-groups hold partial sums of the same 128 x 128 wave tile: each keeps the columns j = 0, 1 and sends 2, 3 through LDS
        u32x4* xbuf = e2m3_smem;
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int qv = 0; qv < 4; ++qv) {
                    const f32x16& t = acc[i][2 + jj];
                    const f32x4 v = {t[qv * 4], t[qv * 4 + 1], t[qv * 4 + 2], t[qv * 4 + 3]};
                    xbuf[((((wn * 2 + (1 - kg)) * IM + i) * 2 + jj) * 4 + qv) * 64 + lane] = __builtin_bit_cast(u32x4, v);
                }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int qv = 0; qv < 4; ++qv) {
                    const f32x4 v = __builtin_bit_cast(f32x4, xbuf[((((wn * 2 + kg) * IM + i) * 2 + jj) * 4 + qv) * 64 + lane]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][jj][qv * 4 + e] += v[e];
                }
        __syncthreads();                                    // the output slabs lie over the exchange
    }

    // Epilogue: lane l, register v -> column (v / 4) * 8 + (l / 32) * 4 + v % 4 of the B tile, token l % 32
    int ln = lane;
    asm volatile("" : "+v"(ln));                           // (addresses are computed here, not kept over the tiles: registers are full)
    const int kh = ln >> 5;
    constexpr int JO = KG == 2 ? 2 : 4;                     // column groups that this wave puts out
    if constexpr (DEQ) {
        // one slab of 32 x 64 behind the other, the stores of each behind the next one's arithmetic
        char* const region = (KG == 1 ? (char*)(colsum + 256) : lds) + wave * 4096;
        const SlabOut out = slab_out(Y, at.m0, M - at.m0 < BM ? M - at.m0 : BM, N, ln);
        Slab slab;
#pragma unroll
        for (int jb = 0; jb < JO; jb += 2) {
            f16x4 sbh[2][4], bih[2][4];
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const int col = wn * 128 + gb(jb + jj) * 32 + gq * 8 + kh * 4;
                    sbh[jj][gq] = *(const f16x4*)(scales + col);
                    bih[jj][gq] = *(const f16x4*)(scales + 256 + col);
                }
#pragma unroll
            for (int i = 0; i < IM; ++i) {
                const f16 sa = scales[512 + wm * TM + ga(i) * 32 + (ln & 31)];
                f16x4 o[2][4];
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    // (moved out of its registers here, not before; what the K-groups have added up is in vector registers already)
                    if constexpr (KG == 1) asm volatile("" : "+a"(acc[i][jb + jj]));
                    else asm volatile("" : "+v"(acc[i][jb + jj]));
#pragma unroll
                    for (int gq = 0; gq < 4; ++gq)
                        o[jj][gq] = dequant4_f32x64(acc[i][jb + jj][gq * 4], acc[i][jb + jj][gq * 4 + 1], acc[i][jb + jj][gq * 4 + 2],
                                                    acc[i][jb + jj][gq * 4 + 3], sa, sbh[jj][gq], bih[jj][gq]);
                }
                if (jb + i > 0)
                    slab_store(out, slab, N, wm * TM + ga(i > 0 ? i - 1 : IM - 1) * 32, at.n0 + wn * 128 + gb(i > 0 ? jb : jb - 2) * 32, ln);
                slab = slab_turn(region, o, ln);
            }
        }
        slab_store(out, slab, N, wm * TM + ga(IM - 1) * 32, at.n0 + wn * 128 + gb(JO - 2) * 32, ln);
    } else {
    // int32 sums: four columns of a row per lane and store
    const int m0 = __builtin_amdgcn_readfirstlane(at.m0);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(C + (int64_t)m0 * N), 0, (int)((u32)(M - m0 < BM ? M - m0 : BM) * (u32)N * 4u), 0x00020000);
#pragma unroll
    for (int i = 0; i < IM; ++i) {
        const u32 row = (u32)(wm * TM + ga(i) * 32 + (ln & 31)) * (u32)N;
#pragma unroll
        for (int j = 0; j < JO; ++j) {
            if constexpr (KG == 1) asm volatile("" : "+a"(acc[i][j]));
            else asm volatile("" : "+v"(acc[i][j]));
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int col = at.n0 + wn * 128 + gb(j) * 32 + gq * 8 + kh * 4;
                const u32 off = (row + (u32)col) * 4u;
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (u32)(int)(64.f * acc[i][j][gq * 4 + e]);
                if ((N & 3) == 0) {                         // (then the four columns exist, and are aligned)
                    __builtin_amdgcn_raw_buffer_store_b128(o, rsrc, col < N ? off : 0xFFFFFF00u, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        __builtin_amdgcn_raw_buffer_store_b32(o[e], rsrc, col + e < N ? off + 4u * e : 0xFFFFFF00u, 0, 0);
                }
            }
        }
    }
    }
    if (KG == 2 || last) return;
    // the next tile's scales into the other half of their place (a slower wave may still read this tile's)
    scales = scales == (f16*)(lds + NBUF * STAGE) ? scales + 512 + BM : (f16*)(lds + NBUF * STAGE);
    park_scales();
    more = false;
    at = then;
    ++t;
    }
#undef QR_E2M3_BARRIER
}

// Tiles are dealt to the XCDs in runs of `per_xcd`, and workgroup b takes every (gridDim / nxcd)-th of its XCD's run
template <bool DEQ, bool RAGGED, int BM>
__global__ __launch_bounds__(256) void gemm_sp256_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int tiles_m, int tiles_n, int nxcd, int) {
    const int tiles = tiles_m * tiles_n, per_xcd = (tiles + nxcd - 1) / nxcd, xcd = blockIdx.x % nxcd;
    const int run = tiles - xcd * per_xcd < per_xcd ? tiles - xcd * per_xcd : per_xcd;
    const int first = blockIdx.x / nxcd, step = gridDim.x / nxcd;
    if (first >= run) return;
    e2m3_tiles<DEQ, RAGGED, BM, 1>(A, B, M, N, Kb, C, Y, sA, sB, bias, (run - first + step - 1) / step, [=](int t) {
        const TilePlace p = tile_place(xcd * per_xcd + first + t * step, tiles_m, tiles_n);
        return Origin{p.tm * BM, p.tn * 256};
    });
}

template <bool DEQ, bool RAGGED>
__global__ __launch_bounds__(256) void gemm_spk_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int tiles_m, int tiles_n, int nxcd, int) {
    const int per_xcd = gridDim.x / nxcd;
    const int tile = (blockIdx.x % nxcd) * per_xcd + blockIdx.x / nxcd;
    if (tile >= tiles_m * tiles_n) return;
    const TilePlace p = tile_place(tile, tiles_m, tiles_n);
    e2m3_tiles<DEQ, RAGGED, 128, 2>(A, B, M, N, Kb, C, Y, sA, sB, bias, 1, [=](int) { return Origin{p.tm * 128, p.tn * 256}; });
}

// Whole rounds of 256x256 tiles over the CUs, then the tiles of the last round, where they are at most half as many as
// there are CUs, as two 128x256 tiles each: a last round of R tiles keeps cus - R CUs idle for a whole tile's time, its halves
// fill 2 R CUs for a part of it.  A workgroup per CU (both kinds need a CU to themselves: LDS): `whole` tiles among them all, a multiple of
// their number, then at most one half each.
template <bool DEQ, bool RAGGED>
__global__ __launch_bounds__(256) void gemm_sp256_tail_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, int M, int N, int Kb, int32_t* __restrict__ C,
    f16* __restrict__ Y, const f16* __restrict__ sA, const f16* __restrict__ sB, const f16* __restrict__ bias,
    int tiles_m, int tiles_n, int nxcd, int whole) {
    const int grid = gridDim.x, b = blockIdx.x;
    e2m3_tiles<DEQ, RAGGED, 256, 1>(A, B, M, N, Kb, C, Y, sA, sB, bias, whole / grid, [=](int t) {
        const int v = b + t * grid;
        const TilePlace p = tile_place((v % nxcd) * (whole / nxcd) + v / nxcd, tiles_m, tiles_n);
        return Origin{p.tm * 256, p.tn * 256};
    });
    const int halves = ((tiles_m * tiles_n - whole) * 2 + nxcd - 1) / nxcd * nxcd;
    const int unit = (b % nxcd) * (halves / nxcd) + b / nxcd;
    if (b >= halves || whole + unit / 2 >= tiles_m * tiles_n) return;
    const TilePlace p = tile_place(whole + unit / 2, tiles_m, tiles_n);
    const int m0 = p.tm * 256 + (unit & 1) * 128;
    if (m0 >= M) return;
    __syncthreads();                                        // the LDS changes hands
    e2m3_tiles<DEQ, RAGGED, 128, 2>(A, B, M, N, Kb, C, Y, sA, sB, bias, 1, [=](int) { return Origin{m0, p.tn * 256}; });
}

}  // namespace

// shape 0 / 1 / 2: tiles of 128 / 192 / 256 rows; 3: 256-row tiles and a last round of 128-row ones (more than one round of tiles, CUs a
// multiple of the XCDs).  Y == nullptr: int32 sums to C.  K up to 131008; operands below 4 GiB (32-bit buffer offsets),
// outputs within qr_e2m3_reach.
int qr_internal_gemm_e2m3(int shape, const void* A, const void* B, int M, int N, int Kb, void* C, void* Y, const void* sA,
                          const void* sB, const void* bias, hipStream_t st) {
    const int bm = shape == 0 ? 128 : shape == 1 ? 192 : 256;
    if ((int64_t)M * Kb >= (1LL << 32) || (int64_t)N * Kb >= (1LL << 32) || !qr_e2m3_reach(bm, N, Y != nullptr))
        return QR_E_UNSUPPORTED;                            // (the dispatcher routes these away)
    const int tiles_m = (M + bm - 1) / bm, tiles_n = (N + 255) / 256;
    const int nxcd = qr_device().xcds, cus = qr_device().cus;
    const int64_t tiles = (int64_t)tiles_m * tiles_n, whole = shape == 3 ? tiles / cus * cus : 0;
    // the grid is a whole number of rounds over the XCDs; 192- and 256-row tiles: a workgroup per CU, which takes several (where K is more
    // than the one stage in which a turn cannot be prepared)
    const bool turns = shape != 0 && Kb > 128 && cus % nxcd == 0;
    if (shape == 3 && (!turns || whole == 0 || 2 * (tiles - whole) > cus)) return QR_E_UNSUPPORTED;      // (mid_plan's rule)
    const int64_t all = (tiles + nxcd - 1) / nxcd * nxcd, grid = turns && all > cus ? cus : all;
    if (grid > 0x3fffffff) return QR_E_SHAPE;
    using Kern = void (*)(const uint8_t*, const uint8_t*, int, int, int, int32_t*, f16*, const f16*, const f16*, const f16*, int, int,
                          int, int);
    // (int32 sums take the kernels for any K)
    static const Kern table[4][3] = {
        {gemm_spk_kernel<true, false>, gemm_spk_kernel<true, true>, gemm_spk_kernel<false, true>},
        {gemm_sp256_kernel<true, false, 192>, gemm_sp256_kernel<true, true, 192>, gemm_sp256_kernel<false, true, 192>},
        {gemm_sp256_kernel<true, false, 256>, gemm_sp256_kernel<true, true, 256>, gemm_sp256_kernel<false, true, 256>},
        {gemm_sp256_tail_kernel<true, false>, gemm_sp256_tail_kernel<true, true>, gemm_sp256_tail_kernel<false, true>}};
    constexpr int lds256 = e2m3_lds(256, 1), lds128 = e2m3_lds(128, 2);
    const size_t lds = shape == 0 ? lds128 : shape == 1 ? e2m3_lds(192, 1) : shape == 2 ? lds256 : lds128 > lds256 ? lds128 : lds256;
    const Kern kern = table[shape][!Y ? 2 : (Kb & 127) != 0 ? 1 : 0];
    const hipError_t e = qr_allow_dynamic_lds((const void*)kern, lds);
    if (e != hipSuccess) return (int)e;
    kern<<<dim3((unsigned)grid), dim3(256), lds, st>>>((const uint8_t*)A, (const uint8_t*)B, M, N, Kb, (int32_t*)C, (f16*)Y,
                                                       (const f16*)sA, (const f16*)sB, (const f16*)bias, tiles_m, tiles_n, nxcd,
                                                       (int)whole);
    return qr_launch_status();
}
