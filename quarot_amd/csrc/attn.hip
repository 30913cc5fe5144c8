// Paged int4 KV cache: appending quantised vectors to their pages, and single-query (decode) attention
// over the cache with the dequantisation done in registers.
#include "qr_kvq.h"

namespace {

// ---- append: pure data movement --------------------------------------------------------------------
// One 16-byte piece per thread: four threads move the 64 code bytes of a (token, head) vector of K and of
// V; the first of them also moves the two {scale, zero} words.
__global__ __launch_bounds__(256) void paged_append_i4_kernel(PagedKV c, const u32x4* __restrict__ key,
                                                              const u32x4* __restrict__ value,
                                                              const u32* __restrict__ kparam, const u32* __restrict__ vparam,
                                                              const int32_t* __restrict__ append_indptr, int64_t tokens) {
    const int64_t pieces = tokens * c.num_heads * 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < pieces; i += (int64_t)gridDim.x * 256) {
        const int piece = (int)(i & 3);
        const int64_t vec = i >> 2, token = vec / c.num_heads;
        const int head = (int)(vec - token * c.num_heads);
        int64_t page;
        int entry;
        if (!paged_locate(c, append_indptr, token, page, entry)) continue;
        const int64_t ks = paged_slot(c, page, 0, head, entry), vs = paged_slot(c, page, 1, head, entry);
        ((u32x4*)c.data)[ks * 4 + piece] = key[i];
        ((u32x4*)c.data)[vs * 4 + piece] = value[i];
        if (piece == 0) {
            c.param[ks] = kparam[vec];
            c.param[vs] = vparam[vec];
        }
    }
}

// ---- decode attention --------------------------------------------------------------------------------
// o[b, h, :] = sum_j softmax_j( q[b, h, :] . k_j / sqrt(128) ) v_j over the sequence's cached vectors, with
// k_j[i] = float(code) * scale_j - zero_j formed in fp32 (quantization.cuh:59-84, decode.cuh:492-689).
// HBM-bound: 128 code bytes + 8 parameter bytes per cached position and head.
//
// A workgroup of four waves serves one (sequence, head) -- or one of `splits` interleaved parts of it.
// A wave takes 16 consecutive positions per step, four lanes per position, so that a lane's 16-byte load
// is one quarter (32 dimensions) of a K or V vector and a wave's load instruction covers 1 KB of
// consecutive cache bytes.  Because  q . k_j = scale_j (q . codes_j) - zero_j sum(q)  the inner loop works on
// the codes themselves: byte-to-float conversions of the masked nibbles (the high nibbles come out
// times 16: folded into the multiplier) and one fma per element, in fp32.  Every group of four lanes
// keeps its own running maximum, denominator and 32-dimension accumulator for the positions it visits
// (U of them per step, so the accumulator is rescaled once per U positions); the 64 partial states of
// the workgroup are merged through LDS at the end.
constexpr int AU = 2;                 // positions per lane group and step (two steps are in flight)

__device__ __forceinline__ float quad_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));   // lanes ^ 1
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));   // lanes ^ 2
    return v;
}

// float(byte k of w): one instruction each (v_cvt_f32_ubyte0..3).  Spelled as asm because the compiler,
// seeing the nibble mask applied before, prefers a 4-bit field extract per element plus ubyte0, which
// doubles the instruction count of the inner loops.
__device__ __forceinline__ float byte_f32(u32 w, int k) {
    float f;
    switch (k) {
        case 0: asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(w)); break;
        case 1: asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(w)); break;
        case 2: asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(w)); break;
        default: asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(w)); break;
    }
    return f;
}

// Codes of one 32-bit word (eight nibbles) as four fp16 pairs, exponent bits or-ed in so that no integer
// to float conversion is needed: pair i holds codes i and i + 4 as BIAS + code, BIAS = 1024 for i = 0, 2
// (code in mantissa bits 0..3 under exponent 25) and 64 for i = 1, 3 (code in mantissa bits 4..7 under
// exponent 21).  One shift and four and-or instructions per word.
struct CodePairs {
    u32 p[4];
};
__device__ __forceinline__ CodePairs code_pairs(u32 w, u32 mask_lo, u32 bias_lo, u32 mask_hi, u32 bias_hi) {
    CodePairs r;
    const u32 w8 = w >> 8;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r.p[0]) : "v"(w), "v"(mask_lo), "v"(bias_lo));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r.p[1]) : "v"(w), "v"(mask_hi), "v"(bias_hi));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r.p[2]) : "v"(w8), "v"(mask_lo), "v"(bias_lo));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r.p[3]) : "v"(w8), "v"(mask_hi), "v"(bias_hi));
    return r;
}
constexpr float kBiasEven = 1024.0f, kBiasOdd = 64.0f;

template <int CTRL>
__device__ __forceinline__ float row_rotate(float v) {   // DPP row_ror within each row of 16 lanes
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// value held by lane (id ^ MASK), for the butterflies of the query's transform
template <int MASK>
__device__ __forceinline__ float butterfly(float t, int lane) {
    // upper lane of a pair: partner - own, lower lane: own + partner
    if constexpr (MASK == 16 || MASK == 32) {
        const u32 w = __builtin_bit_cast(u32, t);
        float lo, hi;
        if constexpr (MASK == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(w, w, false, false);
            lo = __builtin_bit_cast(float, (u32)r[0]), hi = __builtin_bit_cast(float, (u32)r[1]);
        } else {
            const auto r = __builtin_amdgcn_permlane32_swap(w, w, false, false);
            lo = __builtin_bit_cast(float, (u32)r[0]), hi = __builtin_bit_cast(float, (u32)r[1]);
        }
        return (lane & MASK) ? lo - hi : lo + hi;
    } else {
        const int i = __builtin_bit_cast(int, t);
        int o;
        if constexpr (MASK == 1) o = __builtin_amdgcn_mov_dpp(i, 0xB1, 0xF, 0xF, true);
        else if constexpr (MASK == 2) o = __builtin_amdgcn_mov_dpp(i, 0x4E, 0xF, 0xF, true);
        else if constexpr (MASK == 4) o = __builtin_amdgcn_ds_swizzle(i, 0x101F);
        else o = __builtin_amdgcn_mov_dpp(i, 0x128, 0xF, 0xF, true);                    // row_ror:8 == xor 8
        const float other = __builtin_bit_cast(float, o);
        return (lane & MASK) ? other - t : t + other;
    }
}

// sum over the two lanes 32 (or 16) apart of two registers at once: the lower lane ends with a's sum, the upper with b's
template <int MASK>
__device__ __forceinline__ float fold_pair(float a, float b) {
    const u32 wa = __builtin_bit_cast(u32, a), wb = __builtin_bit_cast(u32, b);
    if constexpr (MASK == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(wa, wb, false, false);
        return __builtin_bit_cast(float, (u32)r[0]) + __builtin_bit_cast(float, (u32)r[1]);
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(wa, wb, false, false);
        return __builtin_bit_cast(float, (u32)r[0]) + __builtin_bit_cast(float, (u32)r[1]);
    }
}
__device__ __forceinline__ float wave_total(float v) {      // of a value that the four lanes of a group share: sum over groups
    v += row_rotate<0x124>(v);
    v += row_rotate<0x128>(v);
    v = fold_pair<16>(v, v);
    return fold_pair<32>(v, v);
}

// the partial states of one (sequence, head) -> its output; eight states' loads are in flight at a time
__device__ __forceinline__ void merge_states(const float* src, int splits, int dim, f16* o) {
    auto get = [](const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    float M = -5e4f, D = 0.f, O = 0.f;
    for (int s0 = 0; s0 < splits; s0 += 8) {
        float m8[8], d8[8], o8[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float* p = src + (int64_t)(s0 + k < splits ? s0 + k : splits - 1) * 132;
            m8[k] = get(p), d8[k] = get(p + 1), o8[k] = get(p + 4 + dim);
        }
        float top = M;
#pragma unroll
        for (int k = 0; k < 8; ++k) top = __builtin_fmaxf(top, m8[k]);
        const float keep = __builtin_amdgcn_exp2f(M - top);
        D *= keep, O *= keep, M = top;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float w = s0 + k < splits ? __builtin_amdgcn_exp2f(m8[k] - M) : 0.f;
            D = __builtin_fmaf(d8[k], w, D);
            O = __builtin_fmaf(o8[k], w, O);
        }
    }
    o[dim] = (f16)(O / D);
}

// ALIGNED: page_size is a multiple of 16, so the 16 positions of a wave step lie in one page.
// NW: waves per workgroup (4, 8 or 16): a (sequence, head) gets NW * splits waves in all.
// APPEND: the sequence's LAST position is the token of this step, and its key and value arrive as fp16 vectors
// (knew, vnew: [batch, heads, 128]) instead of lying in the cache already: the last two waves of the (sequence, head), which
// have no more of the cache to walk than the others and often less, quantise the key and the value (kv_quant_one_vector: the
// bits of the quantise-and-append kernel) while their first loads are on the way, write codes and
// parameters to the position's page slot, and leave the position's logit and its dequantised value in LDS as one more
// softmax state for the merge; the walk over the cache stops one position short.  A decode step is then ONE launch
// instead of append + attention.
// Short sequences and small batches are bound by the fixed path of a workgroup, so it is kept short: every load that
// depends on nothing but the workgroup's number (query, new key and value) is requested first, then the first step of the
// cache; a wave transforms the query once, two values per lane (56 vector instructions instead of ~450 with 32 values in
// every lane), and hands it to its lane groups through 256 bytes of LDS; at the end a wave folds its 16 lane groups into
// one state by exchanging halves (64 instructions instead of 190 for four states), so one barrier and a merge of NW
// states remain.
template <bool ALIGNED, int NW, bool APPEND = false>
__global__ __launch_bounds__(64 * NW, (NW == 16 ? 1 : NW == 8 ? 2 : 4)) void paged_decode_i4_kernel(
    const f16* __restrict__ q, uint64_t indptr_at, uint64_t last_page_offset_at, uint64_t indices_at,
    const u32x4* __restrict__ knew, const u32x4* __restrict__ vnew, u32 heads_inverse, u32 page_inverse, u32 shifts, PagedKV c, f16* __restrict__ o,
    float sm_scale_log2, float* __restrict__ part, int had, u32* __restrict__ arrived) {
    // (the arguments that the first loads wait for stand first: they arrive with the waves.  The page tables' addresses come as numbers: for
    // every argument that is a pointer the launch looks its allocation up, 0.06 us each on the host, which bounds the smallest steps)
    using Ints = const __attribute__((address_space(1))) int32_t*;
    const Ints indptr = (Ints)indptr_at, last_page_offset = (Ints)last_page_offset_at, indices = (Ints)indices_at;
    __shared__ f32x4 st4[NW * 33];                         // per wave: [m, d, -, -], 128 outputs; before that the query (256 bytes)
    __shared__ u32x4 fresh[APPEND ? 2 * 16 : 1];           // APPEND: staging of the quantising waves, then the key's codes
    __shared__ float newv[APPEND ? 128 + 2 : 1];           // APPEND: the new position's value and its [m, d]
    float* const st = (float*)st4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = lane >> 2, c4 = lane & 3;
    const int q_had = had & 1, k_had = had >> 1;            // whether the query and the new key are transformed
    const int splits = 1 << (shifts & 31), bh = blockIdx.x >> (shifts & 31), sp = blockIdx.x & (splits - 1);
    const int b = (int)(__umulhi((u32)bh << 2, heads_inverse) >> (shifts >> 16)), h = bh - b * c.num_heads;
    const u32 qword = ((const u32*)q)[(int64_t)bh * 64 + lane];          // dimensions 2 lane, 2 lane + 1
    const bool owns_new = APPEND && sp == splits - 1;       // uniform; of this workgroup's waves the last: the key, the last but one: the value
    const bool appends = owns_new && wave >= NW - 2;
    u32x4 piece = {0, 0, 0, 0};
    if (APPEND && appends) piece = (wave == NW - 1 ? knew : vnew)[(int64_t)bh * 16 + (lane & 15)];
    const int p0 = indptr[b], npages = indptr[b + 1] - p0;
    int last = last_page_offset[b];
    asm volatile("" : "+s"(last));                          // (requested along with the others, not behind the look at npages)
    const int seq_all = npages > 0 ? (npages - 1) * c.page_size + last : 0;
    const int seq_len = APPEND ? seq_all - 1 : seq_all;     // positions read from the cache
    if (npages <= 0) {
        // A sequence without pages (uniform over the workgroups of the pair): nothing may be read -- its slice of kv_indices
        // is empty, and so may be the whole list and the page pool.  The result is the empty softmax state, i.e. the
        // 0 / 0 that the loop below would arrive at (and the reference's kernel does).
        if (threadIdx.x < 128) {
            if (splits == 1 || arrived) {
                o[(int64_t)bh * 128 + threadIdx.x] = (f16)__builtin_nanf("");
            } else {
                float* dst = part + (int64_t)blockIdx.x * 132;
                if (threadIdx.x == 0) {
                    dst[0] = -5e4f;
                    dst[1] = 0.f;
                }
                dst[4 + threadIdx.x] = 0.f;
            }
        }
        return;
    }

    const int chunks = (seq_len + 15) >> 4;
    // a vector's place: slot = page * page_slots + head_slots + entry (K), + kv_slots (V); 64 code bytes and
    // one parameter word per slot
    const int64_t page_slots = (int64_t)c.num_layers * 2 * c.num_heads * c.page_size;
    const int64_t head_slots = ((int64_t)c.layer_idx * 2 * c.num_heads + h) * c.page_size;
    const int64_t kv_slots = (int64_t)c.num_heads * c.page_size;
    const int stride = NW * splits;                         // chunks between the steps of one wave
    // ALIGNED: chunk g lies in page g / cpp at entry 16 (g % cpp); both advance without divisions
    const int cpp = ALIGNED ? c.page_size >> 4 : 1;
    auto pages = [&](int n) { return ALIGNED ? (int)(__umulhi((u32)n << 2, page_inverse) >> (shifts >> 8 & 255)) : n; };       // n / cpp
    const int r_step = stride - pages(stride) * cpp;
    int g = sp * NW + wave;
    // ALIGNED: the page numbers of the wave's next 64 chunks, a lane each (-1: no such page), so that a step takes its own by
    // a lane's number.  (A scalar load in every step, waited for where it stands:
    // 3 x 8000 x 16 heads 16.9 us, now 15.9; 1 x 2048 x 32 8.4, now 8.0; 40 x 438 x 40 26.6, now 25.8.)
    const int g_first = g;
    int r_u = g - pages(g) * cpp, n_u = 0;                  // the chunk's place in its page, and its number among this wave's
    auto fetch_pages = [&](int n) {
        const int it = pages(g_first + (n + lane) * stride);
        const int page = indices[p0 + (it < npages ? it : 0)];
        return it < npages && page >= 0 && page < c.num_pages ? page : -1;
    };
    int page64 = ALIGNED ? fetch_pages(0) : 0;
    // Two sets of AU positions per lane group: the loads of the next set are issued before the current
    // one is consumed, so their latency hides under the arithmetic.  Loads are unconditional (a position
    // beyond the sequence reads entry 0 of a valid page and is masked), which keeps the loop free of
    // branches around memory operations.
    struct Step {
        u32x4 kw[AU], vw[AU];
        u32 kp[AU], vp[AU];
        bool ok[AU];
    };
    auto issue = [&](Step& t, int g0) {
        int64_t page[AU];
        int entry[AU];
        // page numbers first, then every vector load of the step
#pragma unroll
        for (int u = 0; u < AU; ++u) {
            const int pos = (g0 + u * stride) * 16 + slot;
            if (ALIGNED) {
                page[u] = __builtin_amdgcn_readlane(page64, (n_u + u) & 63);        // (wave-uniform)
                entry[u] = r_u * 16 + slot;
                r_u += r_step;
                if (r_u >= cpp) r_u -= cpp;
                t.ok[u] = pos < seq_len;
            } else {
                const int it = pos / c.page_size;
                entry[u] = pos - it * c.page_size;
                t.ok[u] = pos < seq_len && it < npages;
                page[u] = indices[p0 + (it < npages ? it : 0)];
            }
        }
        if (ALIGNED) {
            n_u += AU;
            if ((n_u & 63) == 0) {                          // (and waited for here, not at the next step)
                page64 = fetch_pages(n_u);
                asm volatile("" : "+v"(page64));
            }
        }
#pragma unroll
        for (int u = 0; u < AU; ++u) {
            const bool page_ok = page[u] >= 0 && (ALIGNED || page[u] < c.num_pages);
            t.ok[u] = t.ok[u] && page_ok;
            // the page part of the address is wave-uniform when ALIGNED (scalar base, 32-bit lane offsets)
            const int64_t kbase = (page_ok ? page[u] : 0) * page_slots + head_slots;
            const u32 e = t.ok[u] ? (u32)entry[u] : 0u;
            const uint8_t* kd = c.data + kbase * 64;
            const uint8_t* vd = c.data + (kbase + kv_slots) * 64;
            t.kw[u] = __builtin_nontemporal_load((const u32x4*)(kd + (e * 64u + (u32)c4 * 16u)));
            t.vw[u] = __builtin_nontemporal_load((const u32x4*)(vd + (e * 64u + (u32)c4 * 16u)));
            t.kp[u] = *(const u32*)((const uint8_t*)(c.param + kbase) + e * 4u);
            t.vp[u] = *(const u32*)((const uint8_t*)(c.param + kbase + kv_slots) + e * 4u);
        }
    };
    Step sa, sb;
    int new_page = -1, new_entry = 0;                       // the new token's place
    if (appends) {
        const int pos = seq_all - 1, it = ALIGNED && pos >= 0 ? pages(pos >> 4) : pos / c.page_size;
        new_entry = pos - it * c.page_size;
        // (a scalar load: a vector load's wait would include the first step's, and the quantiser is to run under their latency)
        const Ints from = indices + p0 + __builtin_amdgcn_readfirstlane(it);
        asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=&s"(new_page) : "s"(from) : "memory");
    }
    issue(sa, g);
    __builtin_amdgcn_sched_barrier(0);

    // The query, with the Hadamard over the head dimension (matmul_had_cuda on q, kv_cache.py:30-33,113) here instead of in
    // a launch of its own: 128-point transform in fp32 -- index bit 0 inside the lane, bits 1 .. 6 across lanes -- times
    // 1 / sqrt(128), rounded to fp16 like that function's result.
    // Then this lane's 32 query values as fp16 pairs in the order the codes are consumed: word j of a 16-byte
    // piece holds dimensions 8 j .. 8 j + 7, and (word >> 4 i) & 0x000F000F isolates codes i and i + 4.
    f16x2 qp[4][4];
    float qs, qbias = 0.f;                                 // sum of all 128 values; sum over this lane's of q * (bias of its code)
    {
        u32 w = qword;
        if (q_had) {
            const f16x2 pr = as_f16x2(qword);
            float t0 = (float)pr[0] + (float)pr[1], t1 = (float)pr[0] - (float)pr[1];
            t0 = butterfly<1>(t0, lane), t1 = butterfly<1>(t1, lane);
            t0 = butterfly<2>(t0, lane), t1 = butterfly<2>(t1, lane);
            t0 = butterfly<4>(t0, lane), t1 = butterfly<4>(t1, lane);
            t0 = butterfly<8>(t0, lane), t1 = butterfly<8>(t1, lane);
            t0 = butterfly<16>(t0, lane), t1 = butterfly<16>(t1, lane);
            t0 = butterfly<32>(t0, lane), t1 = butterfly<32>(t1, lane);
            const float hs = 0.08838834764831845f;         // 1 / sqrt(128)
            w = narrow_f16x2(t0 * hs, t1 * hs);
        }
        u32* const mine = (u32*)(st4 + wave * 33);         // private to the wave (LDS operations of one wave execute in order)
        mine[lane] = w;
        __builtin_amdgcn_wave_barrier();
        float ql = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x4 v = ((const u32x4*)mine)[c4 * 4 + j];
#pragma unroll
            for (int k = 0; k < 4; ++k) ql = __builtin_amdgcn_fdot2(as_f16x2(v[k]), f16x2{(f16)1.0f, (f16)1.0f}, ql, false);
            qp[j][0] = as_f16x2(__builtin_amdgcn_perm(v[2], v[0], 0x05040100u));
            qp[j][1] = as_f16x2(__builtin_amdgcn_perm(v[2], v[0], 0x07060302u));
            qp[j][2] = as_f16x2(__builtin_amdgcn_perm(v[3], v[1], 0x05040100u));
            qp[j][3] = as_f16x2(__builtin_amdgcn_perm(v[3], v[1], 0x07060302u));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16 bi = (f16)((i & 1) ? kBiasOdd : kBiasEven);
                qbias = __builtin_amdgcn_fdot2(qp[j][i], f16x2{bi, bi}, qbias, false);
            }
        }
        qs = quad_sum(ql);
        __builtin_amdgcn_wave_barrier();
    }
    u32 mask_lo = 0x000F000Fu, bias_lo = 0x64006400u, mask_hi = 0x00F000F0u, bias_hi = 0x54005400u;
    asm volatile("" : "+v"(mask_lo), "+v"(bias_lo), "+v"(mask_hi), "+v"(bias_hi));     // kept in registers for v_and_or_b32

    // logit of a position from its key's quarter: q . (bias + codes) with fp32 accumulation of exact products, minus
    // sum(q * bias), over the four lanes of the position
    auto logit = [&](u32x4 kw, u32 kp) {
        float a0 = 0.f, a1 = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const CodePairs cp = code_pairs(kw[j], mask_lo, bias_lo, mask_hi, bias_hi);
            a0 = __builtin_amdgcn_fdot2(qp[j][0], as_f16x2(cp.p[0]), a0, false);
            a1 = __builtin_amdgcn_fdot2(qp[j][1], as_f16x2(cp.p[1]), a1, false);
            a0 = __builtin_amdgcn_fdot2(qp[j][2], as_f16x2(cp.p[2]), a0, false);
            a1 = __builtin_amdgcn_fdot2(qp[j][3], as_f16x2(cp.p[3]), a1, false);
        }
        const float dot = quad_sum((a0 + a1) - qbias);
        const f16x2 prm = as_f16x2(kp);
        return (dot * (float)prm[0] - (float)prm[1] * qs) * sm_scale_log2;
    };

    if (APPEND && appends) {
        const bool page_ok = new_page >= 0 && new_page < c.num_pages, key = wave == NW - 1;
        u32x4* const stage = fresh + (key ? 16 : 0);
        const OneVector r = kv_quant_one_vector(piece, stage, key && k_had, 0.08838834764831845f);      // 1 / sqrt(128)
        const u32 prm = pack_scale_zero(r.sc, r.zp);
        if (page_ok) {
            const int64_t s = paged_slot(c, new_page, key ? 0 : 1, h, new_entry);
            c.data[s * 64 + r.at] = (uint8_t)r.byte;
            if (lane == 0) c.param[s] = prm;
        }
        if (key) {
            ((uint8_t*)stage)[r.at] = (uint8_t)r.byte;
            __builtin_amdgcn_wave_barrier();
            const float lg = logit(stage[c4], prm);
            if (lane == 0) {
                newv[128] = page_ok ? lg : -__builtin_inff();
                newv[129] = page_ok ? 1.f : 0.f;
            }
        } else {
            const float z = page_ok ? (float)r.zp : 0.f, s = page_ok ? (float)r.sc : 0.f;
            newv[2 * r.at] = (float)(r.byte & 15u) * s - z;
            newv[2 * r.at + 1] = (float)(r.byte >> 4) * s - z;
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    float m = -5e4f, d = 0.f, pz = 0.f, psum = 0.f, acc[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = 0.f;
    auto consume = [&](const Step& t) {
        float lg[AU], mx = m;
#pragma unroll
        for (int u = 0; u < AU; ++u) {
            const float x = logit(t.kw[u], t.kp[u]);
            lg[u] = t.ok[u] ? x : -__builtin_inff();
            mx = __builtin_fmaxf(mx, lg[u]);
        }
        const float alpha = __builtin_amdgcn_exp2f(m - mx);
        m = mx;
        d *= alpha;
        pz *= alpha;
        psum *= alpha;
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] *= alpha;
#pragma unroll
        for (int u = 0; u < AU; ++u) {
            const float p = __builtin_amdgcn_exp2f(lg[u] - m);
            // (a lane without a position may have fetched the first slot of the page that the new token opens: whatever its
            // memory held, and 0 times a NaN is a NaN.  The codes are finite as they are.)
            const f16x2 prm = as_f16x2(t.ok[u] ? t.vp[u] : 0u);
            const float ps = p * (float)prm[0];
            d += p;
            pz = __builtin_fmaf(p, (float)prm[1], pz);
            psum += ps;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const CodePairs cp = code_pairs(t.vw[u][j], mask_lo, bias_lo, mask_hi, bias_hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // (the even pairs' bias leaves here, exactly, in fp16: sums of 1024 + code are rounded at up to a thousand
                    // times the result.  Two packed instructions more per word, up to 3 % of a step: 1 x 2048 x 32 heads
                    // 8.7 us without and 8.8 with them, 32 x 500 x 32 heads 19.6 and 20.1)
                    f16x2 pr = as_f16x2(cp.p[i]);
                    if ((i & 1) == 0) pr -= f16x2{(f16)kBiasEven, (f16)kBiasEven};
                    acc[8 * j + i] = __builtin_fmaf(ps, (float)pr[0], acc[8 * j + i]);
                    acc[8 * j + i + 4] = __builtin_fmaf(ps, (float)pr[1], acc[8 * j + i + 4]);
                }
            }
        }
    };
    const int gs = stride * AU;
    // Of the waves on a SIMD the oldest is served first: at 32 x 4001 x 8 heads waves 0 .. 3 were through their walk 4.5 us before 4 .. 7,
    // which then had the memory to themselves without the loads in flight that it takes to fill it.  With precedence for the later ones, which
    // also start later, 28.4 -> 27.8 us, 3 x 8000 x 16 heads 15.9 -> 15.6, 7 x 2500 x 16 13.1 -> 12.6.  (By the turns that a wave and
    // its partner have made all end together, and the launch is 2 us longer: in step, both wait for memory and then both compute.)
    const bool late = NW > 4 && wave >= NW / 2;
    if (late) __builtin_amdgcn_s_setprio(1);
    for (; g < chunks; g += 2 * gs) {
        issue(sb, g + gs);
        __builtin_amdgcn_sched_barrier(0);                 // the compiler would otherwise sink the loads below the arithmetic
        consume(sa);
        __builtin_amdgcn_sched_barrier(0);
        issue(sa, g + 2 * gs);
        __builtin_amdgcn_sched_barrier(0);
        if (g + gs < chunks) consume(sb);                  // (no loads inside: the branch does not disturb the wait counts)
        __builtin_amdgcn_sched_barrier(0);
    }
    // ---- merge.  Every lane first takes the remaining bias and the zero points out of its own sums -- sum p (scale code -
    // zero) remains --, so that no step of the merge rounds at the biased sums' magnitude.  (Taken out behind the merge, the
    // even dimensions of 64 positions were off the nearest fp16 value in 26 % of the outputs; in every lane's sums 14 %;
    // with the even bias out of the products 12 %, as the odd dimensions.)
    // Then the wave's 16 lane groups: everything scaled to the wave's maximum and summed -- the outputs by
    // exchanging halves between lanes 32 and 16 apart (a lane of row r of 16 keeps outputs 8 (r & 1) + 16 (r >> 1) .. + 7 of
    // its quarter) and adding up the row's four groups by two rotations.
    {
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] -= (i & 1) ? __builtin_fmaf(psum, kBiasOdd, pz) : pz;
        float M = __builtin_fmaxf(m, row_rotate<0x124>(m));
        M = __builtin_fmaxf(M, row_rotate<0x128>(M));
        const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, M), 0));
        const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, M), 16));
        const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, M), 32));
        const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, M), 48));
        M = __builtin_fmaxf(__builtin_fmaxf(r0, r1), __builtin_fmaxf(r2, r3));
        const float w = __builtin_amdgcn_exp2f(m - M);
        d = wave_total(d * w);
        float v16[16], v8[8];
#pragma unroll
        for (int i = 0; i < 16; ++i) v16[i] = fold_pair<32>(acc[i] * w, acc[i + 16] * w);
#pragma unroll
        for (int i = 0; i < 8; ++i) v8[i] = fold_pair<16>(v16[i], v16[i + 8]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v8[i] += row_rotate<0x124>(v8[i]);
            v8[i] += row_rotate<0x128>(v8[i]);
        }
        f32x4* const mine = st4 + wave * 33;
        if ((lane & 12) == 0) {
            const int base = 1 + c4 * 8 + ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2;
            mine[base] = f32x4{v8[0], v8[1], v8[2], v8[3]};
            mine[base + 1] = f32x4{v8[4], v8[5], v8[6], v8[7]};
        }
        if (lane == 0) mine[0] = f32x4{M, d, 0.f, 0.f};
    }
    __syncthreads();
    // the workgroup's NW states (and the new position's), one thread per dimension
    if (threadIdx.x < 128) {
        const int dim = threadIdx.x;
        float sm_[NW], M = -5e4f;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            sm_[k] = st[k * 132];
            M = __builtin_fmaxf(M, sm_[k]);
        }
        float nm = -__builtin_inff();
        if (owns_new) {
            nm = newv[128];
            M = __builtin_fmaxf(M, nm);
        }
        float D = 0.f, O = 0.f;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const float w = __builtin_amdgcn_exp2f(sm_[k] - M);
            D = __builtin_fmaf(st[k * 132 + 1], w, D);
            O = __builtin_fmaf(st[k * 132 + 4 + dim], w, O);
        }
        if (owns_new) {
            const float w = __builtin_amdgcn_exp2f(nm - M) * newv[129];
            D += w;
            O = __builtin_fmaf(newv[dim], w, O);
        }
        if (splits == 1) {
            o[(int64_t)bh * 128 + dim] = (f16)(O / D);     // an empty sequence gives 0 / 0, as the reference's kernel does
            return;
        }
        // (device scope: past the L2 of this XCD, where the workgroup that merges may not run)
        float* dst = part + (int64_t)blockIdx.x * 132;
        if (dim == 0) {
            __hip_atomic_store(dst, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(dst + 1, D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __hip_atomic_store(dst + 4 + dim, O, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (splits == 1 || !arrived) return;                    // (not merged here: paged_decode_merge_kernel follows)
    // The last of the pair's workgroups to arrive merges their states and leaves the counter at zero for the next launch.
    // Each wave waits until its stores are acknowledged before the barrier, and the count comes behind it.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    __shared__ u32 before;
    if (threadIdx.x == 0) before = __hip_atomic_fetch_add(arrived + bh, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (before != (u32)splits - 1u) return;
    if (threadIdx.x == 0) __hip_atomic_store(arrived + bh, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < 128) merge_states(part + (int64_t)bh * splits * 132, splits, threadIdx.x, o + (int64_t)bh * 128);
}

// combines the `splits` partial states of every (sequence, head)
__global__ __launch_bounds__(128) void paged_decode_merge_kernel(const float* __restrict__ part, int splits,
                                                                 f16* __restrict__ o) {
    merge_states(part + (int64_t)blockIdx.x * splits * 132, splits, threadIdx.x, o + (int64_t)blockIdx.x * 128);
}

// page tables of `batch` sequences of `length` tokens each: page i of sequence b is page number i * batch + b
// (quarot/transformers/kv_cache.py:253-275 builds them with nine torch kernels per decode step)
__global__ __launch_bounds__(256) void page_tables_kernel(int batch, int pages, int last, int32_t* __restrict__ indptr,
                                                          int32_t* __restrict__ indices, int32_t* __restrict__ last_page_offset) {
    const int step = gridDim.x * 256, first = blockIdx.x * 256 + threadIdx.x;
    for (int i = first; i < batch * pages; i += step) {
        const int b = i / pages;
        indices[i] = (i - b * pages) * batch + b;
    }
    for (int b = first; b <= batch; b += step) {
        indptr[b] = b * pages;
        if (b < batch) last_page_offset[b] = last;
    }
}

int check_cache(const void* kv_data, const void* kv_param, const void* kv_indptr, const void* kv_indices,
                const void* last_page_offset, int64_t num_pages, int num_layers, int layer_idx, int num_heads,
                int page_size, int head_dim, int64_t batch_size) {
    if (num_pages < 0 || num_layers <= 0 || layer_idx < 0 || layer_idx >= num_layers || num_heads <= 0 || page_size <= 0 ||
        batch_size < 0 || batch_size > 0x7fffffff || head_dim <= 0)
        return QR_E_SHAPE;
    if (head_dim != 128) return QR_E_UNSUPPORTED;          // as the reference's bindings (CHECK_EQ(head_dim, 128))
    if (batch_size == 0) return QR_OK;
    if (num_pages == 0) return QR_E_SHAPE;                 // sequences but no page pool: nothing a page number could name
    if (!kv_data || !kv_param || !kv_indptr || !kv_indices || !last_page_offset) return QR_E_NULL;
    if (((uintptr_t)kv_data & 15) || ((uintptr_t)kv_param & 3)) return QR_E_ALIGN;
    return QR_OK;
}

}  // namespace

// paged_f16.hip: the same argument checks for the cache with fp16 pages
__attribute__((visibility("hidden"))) int qr_internal_check_paged_cache(const void* kv_data, const void* kv_param,
                                                                        const void* kv_indptr, const void* kv_indices,
                                                                        const void* last_page_offset, int64_t num_pages,
                                                                        int num_layers, int layer_idx, int num_heads,
                                                                        int page_size, int head_dim, int64_t batch_size) {
    return check_cache(kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx, num_heads,
                       page_size, head_dim, batch_size);
}

__attribute__((visibility("hidden"))) PagedKV qr_internal_paged_kv(void* kv_data, void* kv_param, const void* kv_indptr,
                                                                    const void* kv_indices, const void* last_page_offset,
                                                                    int64_t num_pages, int num_layers, int layer_idx,
                                                                    int num_heads, int page_size, int64_t batch_size) {
    PagedKV c;
    c.data = (uint8_t*)kv_data;
    c.param = (u32*)kv_param;
    c.indptr = (const int32_t*)kv_indptr;
    c.indices = (const int32_t*)kv_indices;
    c.last_page_offset = (const int32_t*)last_page_offset;
    c.num_pages = num_pages;
    c.num_layers = num_layers;
    c.layer_idx = layer_idx;
    c.num_heads = num_heads;
    c.page_size = page_size;
    c.batch_size = (int)batch_size;
    return c;
}

extern "C" int qr_page_tables(int64_t batch_size, int64_t length, int page_size, void* kv_indptr, void* kv_indices,
                              void* last_page_offset, void* stream) {
    if (batch_size < 0 || length <= 0 || page_size <= 0) return QR_E_SHAPE;
    if (batch_size == 0) return QR_OK;
    const int64_t pages = (length + page_size - 1) / page_size;
    if (batch_size * pages > 0x3fffffff) return QR_E_SHAPE;
    if (!kv_indptr || !kv_indices || !last_page_offset) return QR_E_NULL;
    const int64_t blocks = (batch_size * pages + 255) / 256;
    page_tables_kernel<<<dim3((unsigned)(blocks > 256 ? 256 : blocks)), dim3(256), 0, (hipStream_t)stream>>>(
        (int)batch_size, (int)pages, (int)(length - (pages - 1) * page_size), (int32_t*)kv_indptr, (int32_t*)kv_indices,
        (int32_t*)last_page_offset);
    return qr_launch_status();
}

extern "C" int qr_kv_append_i4(void* kv_data, void* kv_param, const void* kv_indptr, const void* kv_indices,
                               const void* last_page_offset, int64_t num_pages, const void* k, const void* v,
                               const void* k_param, const void* v_param, const void* append_indptr_or_null,
                               int64_t tokens, int num_layers, int layer_idx, int num_heads, int page_size, int head_dim,
                               int64_t batch_size, void* stream) {
    if (tokens < 0) return QR_E_SHAPE;
    const int rc = check_cache(kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx,
                               num_heads, page_size, head_dim, batch_size);
    if (rc != QR_OK) return rc;
    if (batch_size == 0 || tokens == 0) return QR_OK;
    if (!append_indptr_or_null && tokens != batch_size) return QR_E_SHAPE;     // one new token per sequence
    if (!k || !v || !k_param || !v_param) return QR_E_NULL;
    if (((uintptr_t)k & 15) || ((uintptr_t)v & 15) || ((uintptr_t)k_param & 3) || ((uintptr_t)v_param & 3)) return QR_E_ALIGN;
    const PagedKV c = qr_internal_paged_kv(kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers,
                                           layer_idx, num_heads, page_size, batch_size);
    const int64_t pieces = tokens * num_heads * 4;
    int64_t blocks = (pieces + 255) / 256;
    blocks = blocks > 256 * 32 ? 256 * 32 : blocks;
    paged_append_i4_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
        c, (const u32x4*)k, (const u32x4*)v, (const u32*)k_param, (const u32*)v_param, (const int32_t*)append_indptr_or_null,
        tokens);
    return qr_launch_status();
}

namespace {
// Waves of a workgroup and workgroups of a (sequence, head), by an estimate in microseconds fitted to a sweep of 1 .. 40
// sequences x 89 .. 16000 positions x 8 .. 64 heads with every plan forced, when a workgroup's fixed path was longer than it is now (2099 cases of
// the present kernel: the chosen plan costs 1.1 % more than the best, 4 % in one of ten, 26 % at worst, where few heads are split sixteen times
// and eight are better):
//   3.3 for the launch and its first loads, 2.7 / 3.4 / 5.0 per workgroup of 4 / 8 / 16 waves on the busiest CU (query,
//   merge), 1.8 when the states of several workgroups are merged (+ 0.3 for every eight of them), and the walk: 0.37 per
//   chunk of 16 positions for one wave, but no faster than 0.069 per chunk for a CU (its vector units dequantise; 0.093
//   with a single wave per SIMD).
// One sequence of 2048 x 32 heads: 32 workgroups of 8 waves leave 224 CUs idle and are bound by the vector units of the
// others (14.7 us); 256 workgroups of 4 waves, 8 per head: 9.1 us.
struct DecodePlan {
    int nw, splits;
};
DecodePlan decode_plan(int64_t batch_size, int num_heads, int64_t max_seq_len) {
    const int64_t bh = batch_size * num_heads, cus = qr_device().cus;
    if (max_seq_len <= 0) return DecodePlan{bh >= 4 * cus ? 4 : bh >= cus ? 8 : 16, 1};
    const int64_t chunks = (max_seq_len + 15) / 16;
    DecodePlan best{4, 1};
    double t_best = 1e30;
    for (int nw = 4; nw <= 16; nw *= 2)
        for (int s = 1; s <= 32; s *= 2) {
            if (s > 1 && nw * s > chunks) break;            // (a wave without a chunk of its own)
            const double load = (double)(bh * s) / (double)cus;
            const double busiest = load < 4.0 ? (double)((bh * s + cus - 1) / cus) : load;     // (many small workgroups even out)
            const double wave_chunks = (double)((chunks + nw * s - 1) / (nw * s));
            const double cu_chunks = busiest * (double)chunks / s;
            const double walk_wave = 0.37 * wave_chunks, walk_cu = (busiest * nw <= 4.0 ? 0.093 : 0.069) * cu_chunks;
            const double t = 3.3 + busiest * (nw == 4 ? 2.7 : nw == 8 ? 3.4 : 5.0) + (s > 1 ? 1.8 + 0.3 * (s / 8) : 0.0) +
                             (walk_wave > walk_cu ? walk_wave : walk_cu);
            if (t < t_best) {
                t_best = t;
                best = DecodePlan{nw, s};
            }
        }
    return best;
}
// the workspace: one arrival counter per (sequence, head), then the partial states
size_t decode_counter_bytes(int64_t bh) { return ((size_t)bh * 4 + 255) & ~(size_t)255; }
}  // namespace

extern "C" size_t qr_batch_decode_workspace_bytes(int64_t batch_size, int num_heads, int64_t max_seq_len) {
    if (batch_size <= 0 || num_heads <= 0) return 0;
    const int s = decode_plan(batch_size, num_heads, max_seq_len).splits;
    return s > 1 ? decode_counter_bytes(batch_size * num_heads) + (size_t)batch_size * num_heads * s * 132 * sizeof(float) : 0;
}

namespace {
int batch_decode(void* o, const void* q, const void* kv_data, const void* kv_param, const void* kv_indptr,
                 const void* kv_indices, const void* last_page_offset, int64_t num_pages, int num_layers, int layer_idx,
                 int num_heads, int page_size, int head_dim, int64_t batch_size, int64_t max_seq_len, void* workspace,
                 size_t workspace_bytes, void* stream, int q_had, const void* knew = nullptr, const void* vnew = nullptr,
                 int k_had = 0, bool counters_zero = false) {
    const int rc = check_cache(kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx,
                               num_heads, page_size, head_dim, batch_size);
    if (rc != QR_OK) return rc;
    if (batch_size == 0) return QR_OK;
    if (!o || !q) return QR_E_NULL;
    if (((uintptr_t)q & 15) || ((uintptr_t)o & 1)) return QR_E_ALIGN;
    if (batch_size * num_heads > 0x3fffffff / 64) return QR_E_SHAPE;
    const PagedKV c = qr_internal_paged_kv((void*)kv_data, (void*)kv_param, kv_indptr, kv_indices, last_page_offset, num_pages,
                                           num_layers, layer_idx, num_heads, page_size, batch_size);
    DecodePlan plan = decode_plan(batch_size, num_heads, max_seq_len);
    int splits = plan.splits;
    const size_t counters = decode_counter_bytes(batch_size * num_heads);
    if (splits > 1 && (!workspace || ((uintptr_t)workspace & 15) ||
                       workspace_bytes < counters + (size_t)batch_size * num_heads * splits * 132 * sizeof(float)))
        splits = 1;                                        // no room for partial states: one workgroup per (sequence, head)
    float* const part = splits > 1 ? (float*)((char*)workspace + counters) : nullptr;
    u32* const arrived = splits > 1 && counters_zero ? (u32*)workspace : nullptr;
    const float sm = (float)(1.4426950408889634 / __builtin_sqrt((double)head_dim));
    const unsigned grid = (unsigned)(batch_size * num_heads * splits);
    hipStream_t st = (hipStream_t)stream;
    // n / d as a multiplication: for n below 2^30, with s the least for which 2^s reaches d, floor(4 n ceil(2^(30 + s) / d) / 2^(32 + s))
    auto log2_of = [](int64_t d) { return d > 1 ? 64u - (u32)__builtin_clzll((unsigned long long)d - 1) : 0u; };
    auto inverse = [](int64_t d, u32 s) { return (u32)(((1ull << (30 + s)) + (uint64_t)d - 1) / (uint64_t)d); };
    const int64_t page_chunks = page_size % 16 == 0 ? page_size / 16 : 1;
    const u32 heads_log2 = log2_of(num_heads), page_log2 = log2_of(page_chunks);
    const u32 heads_inverse = inverse(num_heads, heads_log2), page_inverse = inverse(page_chunks, page_log2);
    const u32 shifts = log2_of(splits) | page_log2 << 8 | heads_log2 << 16;
#define QR_DECODE(AL, NWV)                                                                                              \
    do {                                                                                                                \
        auto kern = knew ? paged_decode_i4_kernel<AL, NWV, true> : paged_decode_i4_kernel<AL, NWV, false>;              \
        kern<<<dim3(grid), dim3(64 * NWV), 0, st>>>((const f16*)q, (uint64_t)c.indptr, (uint64_t)c.last_page_offset, (uint64_t)c.indices, \
                                                    (const u32x4*)knew, (const u32x4*)vnew, heads_inverse, page_inverse, shifts, c, (f16*)o, sm, part, (q_had ? 1 : 0) | (k_had ? 2 : 0), arrived); \
    } while (0)
    if (page_size % 16 == 0) {
        if (plan.nw == 16) QR_DECODE(true, 16);
        else if (plan.nw == 8) QR_DECODE(true, 8);
        else QR_DECODE(true, 4);
    } else {
        if (plan.nw == 16) QR_DECODE(false, 16);
        else if (plan.nw == 8) QR_DECODE(false, 8);
        else QR_DECODE(false, 4);
    }
#undef QR_DECODE
    int lrc = qr_launch_status();
    if (lrc != QR_OK || splits == 1 || arrived) return lrc;
    paged_decode_merge_kernel<<<dim3((unsigned)(batch_size * num_heads)), dim3(128), 0, st>>>(part, splits, (f16*)o);
    return qr_launch_status();
}
}  // namespace

extern "C" int qr_batch_decode_i4(void* o, const void* q, const void* kv_data, const void* kv_param, const void* kv_indptr,
                                  const void* kv_indices, const void* last_page_offset, int64_t num_pages, int num_layers,
                                  int layer_idx, int num_heads, int page_size, int head_dim, int64_t batch_size,
                                  int64_t max_seq_len, void* workspace, size_t workspace_bytes, void* stream) {
    return batch_decode(o, q, kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx,
                        num_heads, page_size, head_dim, batch_size, max_seq_len, workspace, workspace_bytes, stream, 0);
}

extern "C" int qr_batch_decode_qhad_i4(void* o, const void* q, const void* kv_data, const void* kv_param, const void* kv_indptr,
                                       const void* kv_indices, const void* last_page_offset, int64_t num_pages, int num_layers,
                                       int layer_idx, int num_heads, int page_size, int head_dim, int64_t batch_size,
                                       int64_t max_seq_len, void* workspace, size_t workspace_bytes, void* stream) {
    return batch_decode(o, q, kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx,
                        num_heads, page_size, head_dim, batch_size, max_seq_len, workspace, workspace_bytes, stream, 1);
}

// One decode step in one launch: the new token's key and value (fp16 [batch, heads, 128], one token per sequence, its
// place the LAST position of the sequence as the page tables already count it) are quantised inside the attention kernel
// -- the codes and parameters of qr_kv_quant_append_f16_i4, written to the same page slots -- and attended to along with
// the cached positions: qr_kv_quant_append_f16_i4 followed by qr_batch_decode_i4 / _qhad_i4
// (MultiLayerPagedKVCache4Bit.update and the callable it returns, quarot/transformers/kv_cache.py:104-129,224-251).
extern "C" int qr_kv_quant_append_batch_decode_f16_i4(void* o, const void* q, int q_had_mode, const void* k, const void* v,
                                                      int k_had_mode, void* kv_data, void* kv_param, const void* kv_indptr,
                                                      const void* kv_indices, const void* last_page_offset, int64_t num_pages,
                                                      int num_layers, int layer_idx, int num_heads, int page_size, int head_dim,
                                                      int64_t batch_size, int64_t max_seq_len, void* workspace,
                                                      size_t workspace_bytes, void* stream) {
    const bool counters_zero = (q_had_mode & QR_DECODE_COUNTERS_ZERO) != 0;
    q_had_mode &= ~QR_DECODE_COUNTERS_ZERO;
    if ((q_had_mode != 0 && q_had_mode != 1) || (k_had_mode != 0 && k_had_mode != 1)) return QR_E_DTYPE;
    if (batch_size > 0 && (!k || !v)) return QR_E_NULL;
    if (((uintptr_t)k & 15) || ((uintptr_t)v & 15)) return QR_E_ALIGN;
    return batch_decode(o, q, kv_data, kv_param, kv_indptr, kv_indices, last_page_offset, num_pages, num_layers, layer_idx,
                        num_heads, page_size, head_dim, batch_size, max_seq_len, workspace, workspace_bytes, stream, q_had_mode,
                        k, v, k_had_mode, counters_zero);
}
