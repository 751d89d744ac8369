// dcq_attn_prompt.hip — attention of prompts and prompt chunks over the paged KV cache, on f16 MFMA.
//
// The reference's standard attention path (core/src/inference.cpp:1577-1746) in fp32, for calls with
// many query rows; decode-sized calls keep attn_kernel (dcq_kv.hip). The fp32 MFMA peak is 157
// TFLOP/s, a sixteenth of the f16 one, so each fp32 operand x is split into two f16 pieces,
//   x = 2^e (h + l),  h = f16(x 2^-e),  l = f16(x 2^-e - h)   (round to nearest even)
// and a product takes three MFMAs: h h' + h l' + l h'. Two pieces hold 22 bits or more of x, and the
// dropped l l' is below 2^-22 of the product. The exponents keep the pieces in f16's range for every fp32
// input: one per query row, and one per 8 keys for K and for V (the wave that stages 8 keys finds
// their largest magnitude), chosen so that the largest magnitude lands in [2^14, 2^15). An element 2^-r of
// it keeps 22 bits or more for r up to 16, 39 - r beyond.
//
// Work split. The query rows of a KV head are the (token, query head of its group) pairs, token-major,
// so any group size fills the tiles: a workgroup takes 128 consecutive rows, each of its 4 waves 32 of
// them (one column of MFMA tiles), and walks the keys its rows see in blocks of 32, double-buffered in
// LDS. The staging of a block (loads, exponents, split) is shared by the 128 rows; its loads are issued
// before the previous block's MFMAs and its conversion runs after them.
//   At head_dim 128 a workgroup is two such groups of 4 waves over the same rows, alternate blocks each, and
//   fills its CU; the second group's sums are added through LDS at the end. As two workgroups of a CU, a
//   long tile outlived the short one beside it and ran one wave a SIMD, 2.9 us a block against 4.1 us for two
//   blocks together. The second group converts its next block before its MFMAs, the first after them: one
//   group's VALU phase meets the other's MFMAs, though both wait at the same barriers. 2048 tokens, 32/8
//   heads: 198 us as two workgroups, 167 as two groups, 154 with the second one's order turned; 512 tokens
//   over 4096 keys 161, 156, 152 (events over 20 calls of two KV writes and the attention).
//   S^T = K Q^T (keys x rows): A = K pieces (16-byte LDS reads), B = Q pieces (registers). Lane l then
//   holds keys 8 (i/4) + 4 (l/32) + i%4, i = 0..15, of row l%32: the row's softmax is lane-local but for
//   one exchange with the other half-wave, and i/4 is the 8-key group whose exponents apply.
//   O^T += V^T P^T (dims x rows): A = V^T pieces by transposing LDS reads (ds_read_b64_tr_b16), B = the
//   lane's own weights split into pieces, so P is never moved between lanes.
// The softmax weight of a key carries its V exponent, p' = 2^(s + ev - m), so that 2^7 p' V 2^-ev are the
// terms of O; the running reference m is an integer, raised only when the maximum passes it by 8
// (2^7 p' <= 2^15), so O is rescaled a few times per row, and s + (ev - m) is one fma of the MFMA's sum.
// The sum of weights is that of p' 2^-ev, which holds while the exponents ev of a row's keys are within 80
// octaves (kEvMin .. kEvMax, keys of zeros at the lower end): a key as probable as the row's best then has
// p' >= 2^-82.
// Wide groups. One exponent for 8 keys costs a key bits where another is far larger, be it one that the row
// does not see. Keys of a group more than kSpread octaves apart get an exponent each, and such a group, or
// one of values outside kEvMin .. kEvMax, is staged a second time with the exponent kWide, whose sum with
// any score asks for a new reference. From there on the wave takes each key's exponents and sums the weights
// against a reference of their own, straight from the scores (one exp2 more per weight). Ordinary groups
// pay for the test of their spread and a branch that is not taken: 2048 tokens 141 -> 145 us, 333 tokens
// over 2777 keys 63 -> 64 (a per-key exponent throughout: 151 and 66).
//
// Roundings. What is left of the error is the sums', and the scores' most of it: a rounding at a score of 8
// moves its weight by 8 x 2^-25. So a score's small products are added up first, where their roundings are
// small too, and the 8 or 16 h h' MFMAs of head_dim 128 and 256 in two sums; the exponent of a weight near
// the reference is near 0 when it is rounded (2^7 is a factor of the pieces, not of p'); and at head_dim 256
// a block's terms of O are added to it in one rounding. Relative 2-norm error against 64 bits, VALU or fp32
// MFMA kernel before / this kernel with one chain for each sum / as it is: 2048 tokens, 32/8 heads x 128,
// Q8_0: 9.2e-7 / 5.4e-7 / 3.5e-7; 4 tokens over 4095 keys 4.7e-7 / 7.5e-7 / 3.8e-7; 333 tokens over 2777 keys
// x 64, F16: 8.9e-7 / 4.6e-7 / 4.0e-7; x 256, 8 tokens over 8000 keys 4.4e-7 / 1.02e-6 / 4.2e-7, 2048 tokens
// 3.9e-7 / 7.5e-7 / 3.4e-7. Cost, the same calls: 162 -> 166 us, 24.1 -> 24.6, 72.4 -> 72.6, 59.8 -> 62.6,
// 402 -> 425 (events over 20 calls of two KV writes and the attention).
//
// Measured (MI355X), this kernel against the fp32 MFMA one it replaces: a 2048-token prompt, 32/8 heads
// x 128, 377 -> 148 us; 333 tokens over 2777 keys, 32/8 heads x 64, F16, 139 -> 64 us.
#include "dcq_common.h"
#include "dcq_kernels.h"
#include "dcq_attn.h"

namespace dcq {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kBlk = 32;        // keys per block
constexpr int kRows = 128;      // query rows per workgroup
constexpr float kPScale = 128.0f;  // of the weights' pieces: 2^7 at their row's reference, 2^15 before it is raised
constexpr int kEBias = 141;     // exponent field of a group's largest magnitude - its exponent: 127 + 14
constexpr int kEvMin = -64, kEvMax = 16;  // values of 2^-50 .. 2^31
constexpr int kEvZero = kEvMin - 1;       // of a group of zeros, kEvFloor where the keys' own exponents count:
constexpr int kEvFloor = 30 - kEBias;     // norm_exp's smallest
constexpr float kWide = 0x1p100f;         // in place of the ev of a group whose keys' own exponents count
constexpr int kSpread = 12;               // octaves that the keys of a group may lie apart under one exponent

// Wave groups of a workgroup: two at head_dim 128. At 256 one group's blocks fill a CU's LDS, and at 64 a CU
// holds three workgroups of one group, which two groups each measured slower (333 tokens over 2777 keys 67.9
// -> 74.3 us, 2048 tokens of 14/2 heads 65.4 -> 88.5).
constexpr int prompt_groups(int hd) { return hd == 128 ? 2 : 1; }

template <int HD>
struct __align__(16) PromptSmem {
    // pitches: K rows are read 16 bytes per lane down a column of 32 rows (4 banks apart); V rows four
    // at a time, 64 bytes each (16 banks apart)
    static constexpr int KP = HD + 8, VP = HD + 32;
    _Float16 k[2][2][kBlk][KP];  // [buffer][piece][key][dim]
    _Float16 v[2][2][kBlk][VP];
    float ks[2][4], ev[2][4], vi[2][4];  // per 8 keys: 2^ek, ev (or kWide), 2^-ev
    float ks1[2][kBlk], ev1[2][kBlk];    // per key, only of wide groups: 2^ek, ev
};

// The exponent field that normalises magnitudes up to m: m * pow2(268 - E) is in [2^14, 2^15).
__device__ __forceinline__ int norm_exp(uint32_t bits) {
    return max((int)(bits >> 23), 30);  // below 2^-97 (zeros too): the floor's exponent
}
__device__ __forceinline__ float pow2_bits(int e) { return __uint_as_float((uint32_t)e << 23); }

// four consecutive fp32 values (already scaled) -> the f16 pieces
__device__ __forceinline__ void split4(const float x0, const float x1, const float x2, const float x3, f16x4& h,
                                       f16x4& l) {
    const f16x2 h0 = __builtin_convertvector((f32x2){x0, x1}, f16x2);
    const f16x2 h1 = __builtin_convertvector((f32x2){x2, x3}, f16x2);
    const f16x2 l0 = __builtin_convertvector((f32x2){x0 - (float)h0[0], x1 - (float)h0[1]}, f16x2);
    const f16x2 l1 = __builtin_convertvector((f32x2){x2 - (float)h1[0], x3 - (float)h1[1]}, f16x2);
    h = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
    l = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
}

// Transposing LDS read, per 16 lanes: lane j gives the address of elements 4 (j % 4) .. + 3 of row j / 4
// of a 4 x 16 matrix and receives column j.
__device__ __forceinline__ f16x4 lds_transposed(const _Float16* src) {
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) i16x4 LdsI16x4;
    return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)src));
}

// One staging thread's E elements of a K (V) row, as loaded: fp32 words of a current row, or the
// slot's words (Q8_0: E / 4 words of quants and the block's scale; F16: E / 2 words).
template <int E>
struct RawRow {
    uint32_t w[E];
    uint32_t d;
};

template <int CT, int E>
__device__ __forceinline__ void load_raw_slot(const uint8_t* head, int e0, RawRow<E>& r) {
    if constexpr (CT == kTypeQ8_0) {
        const uint8_t* b = head + (e0 / 32) * 34;
        r.d = ldu16(b);
        __builtin_memcpy(r.w, b + 2 + e0 % 32, E);  // 2-byte aligned
    } else {
        constexpr int B = CT == kTypeF16 ? 2 : 4;
#pragma unroll
        for (int j = 0; j < B * E / 16; ++j) {
            const uint4 t = ld16(head + B * e0 + 16 * j);
            r.w[4 * j] = t.x, r.w[4 * j + 1] = t.y, r.w[4 * j + 2] = t.z, r.w[4 * j + 3] = t.w;
        }
    }
}

template <int CT, int E>
__device__ __forceinline__ void decode_raw(const RawRow<E>& r, bool hist, float (&x)[E]) {
    if (CT != kTypeF32 && hist) {
        if constexpr (CT == kTypeQ8_0) {
            const float d = half_bits_to_float(r.d);
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = d * (float)(int32_t)__builtin_amdgcn_sbfe(r.w[j / 4], 8 * (j % 4), 8);
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = half_bits_to_float(j % 2 ? r.w[j / 2] >> 16 : r.w[j / 2] & 0xFFFF);
        }
    } else {
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = __uint_as_float(r.w[j]);
    }
}

// The largest of a staging thread's values m >= 0 over its key (8 lanes) and over the wave's 8 keys.
struct KeyMax {
    uint32_t key, group;  // the bits
};
__device__ __forceinline__ KeyMax key_max(float m) {
    int b = (int)__float_as_uint(m);  // non-negative: ordered as integers
    b = max(b, __builtin_amdgcn_update_dpp(b, b, 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    b = max(b, __builtin_amdgcn_update_dpp(b, b, 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
    b = max(b, __builtin_amdgcn_update_dpp(b, b, 0x141, 0xF, 0xF, false));  // row_half_mirror
    const int key = b;
    b = max(b, __builtin_amdgcn_update_dpp(b, b, 0x140, 0xF, 0xF, false));  // row_mirror
    const int s = max(max(__builtin_amdgcn_readlane(b, 0), __builtin_amdgcn_readlane(b, 16)),
                      max(__builtin_amdgcn_readlane(b, 32), __builtin_amdgcn_readlane(b, 48)));
    return {(uint32_t)key, (uint32_t)s};
}

template <int E>
__device__ __forceinline__ KeyMax key_amax(const float (&x)[E]) {
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) m = fmaxf(m, fabsf(x[j]));
    return key_max(m);
}

// The same of the finite elements: an infinity (its own terms are infinite or NaN) must not set the exponent
// of the finite ones beside it, which would flush to zero.
template <int E>
__device__ __forceinline__ KeyMax key_amax_finite(const float (&x)[E]) {
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) m = fmaxf(m, fabsf(x[j]) < INFINITY ? fabsf(x[j]) : 0.0f);
    return key_max(m);
}

// Whether the keys of a group lie too far apart for one exponent (zeros are exact under any): an element
// keeps 39 - r bits when it is 2^-r of what its exponent was chosen for, so within kSpread octaves a key's
// largest keep 27 or more. True also where one holds an infinity.
__device__ __forceinline__ bool uneven_keys(const KeyMax& m) {
    const uint32_t least = (uint32_t)max((int)m.group - (kSpread << 23), 1);
    return __any(m.key - 1u < least - 1u) || m.group == 0x7F800000u;
}

template <int CT, int HD>
__global__ void __launch_bounds__(256 * prompt_groups(HD), HD == 64 ? 3 : 1) attn_prompt_kernel(AttnArgs a) {
    constexpr int G = prompt_groups(HD);
    constexpr int E = HD / 8;    // elements per staging thread
    constexpr int KS = HD / 16;  // k-steps of the score product
    constexpr int NT = HD / 32;  // 32-dim tiles of the output
    constexpr int KC = HD == 64 ? 1 : 2;  // sums of a score's h h' products
    using Smem = PromptSmem<HD>;
    __shared__ Smem smem[G];
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    Smem& sm = smem[grp];
    const int tid = threadIdx.x & 255, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int p = lane >> 5, c32 = lane & 31;
    const int rep = a.n_head / a.n_head_kv;
    const int n_rows = a.n_tokens * rep;
    const int n_qt = (n_rows + kRows - 1) / kRows;
    const int id = blockIdx.x;
    const int h_kv = id % a.n_head_kv;
    const int split = (id / a.n_head_kv) % a.splits;
    // query tiles see more key blocks the later their tokens: largest first, so that the CUs, which take
    // workgroups as they finish, end together. At head_dim 64, where all of an unsplit launch is resident at
    // once, the second half of the order takes the smallest tiles, ascending, so that a CU's workgroups (one
    // from each half, in dispatch order) carry about the same keys together (with splits largest first: 1500
    // tokens over 100 keys, 24/8 heads, 85.3 -> 74.3 us; 2048 tokens, 14/2 heads, 73.0 -> 65.4)
    const int rank = id / a.n_head_kv / a.splits, half = (n_qt + 1) / 2;
    const int qt = HD == 64 && a.splits == 1 && rank >= half ? rank - half : n_qt - 1 - rank;
    const int64_t hb = CT == kTypeQ8_0 ? (int64_t)(HD / 32) * 34 : (int64_t)HD * (CT == kTypeF16 ? 2 : 4);

    // ---- the lane's query row: pieces of q * scale * log2(e) at dims 16 s + 8 p .. + 7
    const int r0 = qt * kRows + 32 * wave;  // the wave's first row
    const int row = r0 + c32;
    const bool q_ok = row < n_rows;
    const int tok = (q_ok ? row : 0) / rep, h = h_kv * rep + (q_ok ? row : 0) % rep;
    f16x8 qh[KS], ql[KS];
    float qsc;
    {
        const float* qp = a.q + (int64_t)tok * a.q_stride + (int64_t)h * HD + 8 * p;
        float qv[KS][8], m = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 t = *reinterpret_cast<const float4*>(qp + 16 * s + 4 * j);
                qv[s][4 * j] = t.x * a.scale_log2e, qv[s][4 * j + 1] = t.y * a.scale_log2e;
                qv[s][4 * j + 2] = t.z * a.scale_log2e, qv[s][4 * j + 3] = t.w * a.scale_log2e;
            }
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(qv[s][j]));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        const int e = norm_exp(__float_as_uint(m));
        const float f = pow2_bits(268 - e);
        qsc = pow2_bits(e - 14);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            f16x4 h0, l0, h1, l1;
            split4(qv[s][0] * f, qv[s][1] * f, qv[s][2] * f, qv[s][3] * f, h0, l0);
            split4(qv[s][4] * f, qv[s][5] * f, qv[s][6] * f, qv[s][7] * f, h1, l1);
            qh[s] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
            ql[s] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }

    // keys 0 .. n_past + last token are visible to some row of the tile; with key splits this
    // workgroup takes blocks [split * cps, split * cps + cps) of them (possibly none)
    const int last_tok = (min((qt + 1) * kRows, n_rows) - 1) / rep;
    const int nblk = (a.n_past + last_tok + kBlk) / kBlk;
    const int b_begin = split * a.cps, b_end = min(nblk, b_begin + a.cps);
    // the wave's rows: keys up to first_vis are visible to all of them, past last_vis to none
    const int first_vis = a.n_past + min(r0, n_rows - 1) / rep;
    const int last_vis = r0 < n_rows ? a.n_past + min(r0 + 31, n_rows - 1) / rep : -1;

    // ---- staging: thread -> key tid / 8 of the block, E elements from se0; wave w stages keys 8w..8w+7
    const int skey = tid >> 3, se0 = E * (tid & 7);
    RawRow<E> rk, rv;
    int kind = 0;  // what rk, rv hold: 0 zeros, 1 history words, 2 fp32 words of a current row
    auto table_of = [&](int bi) {  // the block-table entry of this thread's key in block bi
        const int lb = (kBlk * bi + skey) / 16;
        return kBlk * bi + skey < a.n_past && lb < a.n_table ? a.table[lb] : -1;
    };
    auto load_block = [&](int bi, int blk) {
        const int kk = kBlk * bi + skey;
        kind = 0;
        if (kk < a.n_past) {
            if (blk >= 0 && blk < a.n_blocks) {
                const int64_t off = (((int64_t)blk * a.n_layer + a.layer) * 16 + kk % 16) * a.sb + (int64_t)h_kv * hb;
                load_raw_slot<CT, E>(a.k_arena + off, se0, rk);
                load_raw_slot<CT, E>(a.v_arena + off, se0, rv);
                kind = 1;
            }
        } else if (kk < a.n_past + a.n_tokens) {
            const int64_t off = (int64_t)(kk - a.n_past) * a.kv_stride + (int64_t)h_kv * HD;
            load_raw_slot<kTypeF32, E>(reinterpret_cast<const uint8_t*>(a.k_cur + off), se0, rk);
            load_raw_slot<kTypeF32, E>(reinterpret_cast<const uint8_t*>(a.v_cur + off), se0, rv);
            kind = 2;
        }
    };
    auto store_piece = [&](const float(&x)[E], float f, _Float16* dh, _Float16* dl) {
#pragma unroll
        for (int j = 0; j < E; j += 8) {
            f16x4 h0, l0, h1, l1;
            split4(x[j] * f, x[j + 1] * f, x[j + 2] * f, x[j + 3] * f, h0, l0);
            split4(x[j + 4] * f, x[j + 5] * f, x[j + 6] * f, x[j + 7] * f, h1, l1);
            *reinterpret_cast<f16x8*>(dh + j) = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
            *reinterpret_cast<f16x8*>(dl + j) = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    auto decode = [&](const RawRow<E>& r, float(&x)[E]) {
        if (kind)
            decode_raw<CT, E>(r, kind == 1, x);
        else
#pragma unroll
            for (int j = 0; j < E; ++j) x[j] = 0.0f;
    };
    // the wave's 8 keys under one exponent each for K and V; true if they are a wide group, for commit_wide
    auto commit_block = [&](int buf) {
        float x[E];
        decode(rk, x);
        KeyMax m = key_amax<E>(x);
        bool wide = uneven_keys(m);
        const int ek = norm_exp(m.group);
        store_piece(x, pow2_bits(268 - ek), &sm.k[buf][0][skey][se0], &sm.k[buf][1][skey][se0]);
        if (lane == 0) sm.ks[buf][wave] = pow2_bits(ek - 14);
        decode(rv, x);
        m = key_amax<E>(x);
        wide |= uneven_keys(m);
        const int ev = m.group ? norm_exp(m.group) : kEBias + kEvZero;
        store_piece(x, pow2_bits(268 - ev), &sm.v[buf][0][skey][se0], &sm.v[buf][1][skey][se0]);
        if (lane == 0) {
            sm.ev[buf][wave] = (float)(ev - kEBias);
            sm.vi[buf][wave] = pow2_bits(268 - ev);
        }
        return wide || ev < kEBias + kEvZero || ev > kEBias + kEvMax || (m.group && ev == kEBias + kEvZero);
    };
    // the same keys again, each under its own exponents. An infinity's l would be NaN: its pieces are 0 and
    // itself, of which only l meets one factor alone (h of the other operand), so that its product is
    // infinite of the right sign, or NaN beside a zero, as in fp32
    auto store_wide = [&](const float(&x)[E], int e, _Float16* dh, _Float16* dl) {
        store_piece(x, pow2_bits(268 - e), dh, dl);
#pragma unroll
        for (int j = 0; j < E; ++j)
            if (fabsf(x[j]) == INFINITY) dh[j] = (_Float16)0.0f, dl[j] = (_Float16)x[j];
    };
    auto commit_wide = [&](int buf, int bi) {
        load_block(bi, table_of(bi));
        float x[E];
        decode(rk, x);
        const int ek = norm_exp(key_amax_finite<E>(x).key);
        store_wide(x, ek, &sm.k[buf][0][skey][se0], &sm.k[buf][1][skey][se0]);
        decode(rv, x);
        const int ev = norm_exp(key_amax_finite<E>(x).key);
        store_wide(x, ev, &sm.v[buf][0][skey][se0], &sm.v[buf][1][skey][se0]);
        sm.ks1[buf][skey] = pow2_bits(ek - 14);
        sm.ev1[buf][skey] = (float)(ev - kEBias);
        sm.ev[buf][wave] = kWide;
    };

    f32x16 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[t][v] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;  // l_run: this lane's keys only, until the end
    bool own_ref = false;  // (uniform) from here on the sum of weights is l_own, in units of 2^m_own
    float m_own = -INFINITY, l_own = 0.0f;

    int blk_next = -1;
    const int b0 = b_begin + grp, lead = G == 2 ? grp : 0;  // lead: the group loads one block further ahead
    if (b0 < b_end) {
        load_block(b0, table_of(b0));
        if (b0 + G < b_end) blk_next = table_of(b0 + G);
        if (__builtin_expect(commit_block(0), 0)) commit_wide(0, b0);
        if (lead && b0 + G < b_end) {
            load_block(b0 + G, blk_next);
            if (b0 + 2 * G < b_end) blk_next = table_of(b0 + 2 * G);
        }
    }
    __syncthreads();
    for (int b = b_begin; b < b_end; b += G) {  // the same turns for every group: barriers
        const int bi = b + grp, kb = kBlk * bi, buf = (b - b_begin) / G & 1;
        const bool more = bi + G < b_end;
        const int nb = bi + G * (1 + lead);
        if (lead && more && __builtin_expect(commit_block(buf ^ 1), 0)) commit_wide(buf ^ 1, bi + G);
        if (nb < b_end) {
            load_block(nb, blk_next);
            if (nb + G < b_end) blk_next = table_of(nb + G);
        }
        if (bi < b_end && kb <= last_vis) {
            // ---- S^T = K Q^T: the small products first, then h h' in KC sums of their own
            const _Float16* kh = &sm.k[buf][0][c32][8 * p];
            const _Float16* kl = &sm.k[buf][1][c32][8 * p];
            f32x16 sc;
#pragma unroll
            for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const f16x8 fh = *reinterpret_cast<const f16x8*>(kh + 16 * s);
                const f16x8 fl = *reinterpret_cast<const f16x8*>(kl + 16 * s);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fl, qh[s], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fh, ql[s], sc, 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                f32x16 d;
#pragma unroll
                for (int v = 0; v < 16; ++v) d[v] = c ? 0.0f : sc[v];
#pragma unroll
                for (int s = c * KS / KC; s < (c + 1) * KS / KC; ++s) {
                    const f16x8 fh = *reinterpret_cast<const f16x8*>(kh + 16 * s);
                    d = __builtin_amdgcn_mfma_f32_32x32x16_f16(fh, qh[s], d, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) sc[v] = c ? sc[v] + d[v] : d[v];
            }

            // ---- the online softmax of the lane's row over its 16 keys
            float cj[4], ev[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // finite and above 0 whatever the exponents: a score past either end weighs the same, and
                // the product of two floors (a row and keys of zeros) must not meet the mask as 0 * -inf
                cj[j] = __builtin_amdgcn_fmed3f(sm.ks[buf][j] * qsc, 0x1p-126f, 0x1.fffffep127f);
                ev[j] = sm.ev[buf][j];
            }
            if (kb + kBlk - 1 > first_vis) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    // a masked key: -inf times cj > 0
                    if (kb + 8 * (i >> 2) + 4 * p + (i & 3) > a.n_past + tok) sc[i] = -INFINITY;
                }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, __builtin_fmaf(sc[i], cj[i >> 2], ev[i >> 2]));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            if (own_ref || __any(mx > m_run + 8.0f)) {
                int wide = 0;  // (uniform) bit j: group j is wide
#pragma unroll
                for (int j = 0; j < 4; ++j) wide |= ev[j] == kWide ? 1 << j : 0;
                wide = __builtin_amdgcn_readfirstlane(wide);
                if (__builtin_expect(wide && !own_ref, 0)) {
                    own_ref = true;
                    m_own = m_run, l_own = l_run;
                    // while o is zero its reference is still to choose: that of zeros is far above tiny values
                    float any_o = 0.0f;
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int v = 0; v < 16; ++v) any_o = fmaxf(any_o, fabsf(o[t][v]));
                    if (fmaxf(any_o, __shfl_xor(any_o, 32, 64)) == 0.0f) m_run = -INFINITY;
                }
                if (__builtin_expect(own_ref, 0)) {
                    // the scores themselves, their sum of weights, then the exponents of the terms of O, which
                    // the fma below is to leave as they are
                    const float* ks1 = &sm.ks1[buf][4 * p];
                    const float* ev1 = &sm.ev1[buf][4 * p];
                    float ms = -INFINITY;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        float c = cj[i >> 2];
                        if (wide & (1 << (i >> 2)))
                            c = __builtin_amdgcn_fmed3f(ks1[8 * (i >> 2) + (i & 3)] * qsc, 0x1p-126f, 0x1.fffffep127f);
                        sc[i] *= c;
                        ms = fmaxf(ms, sc[i]);
                    }
                    ms = fmaxf(m_own, __builtin_ceilf(fmaxf(ms, __shfl_xor(ms, 32, 64))));
                    if (ms != -INFINITY) {
                        l_own *= __builtin_amdgcn_exp2f(m_own - ms);
#pragma unroll
                        for (int i = 0; i < 16; ++i) l_own += __builtin_amdgcn_exp2f(sc[i] - ms);
                        m_own = ms;
                    }
                    mx = -INFINITY;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        float e = ev[i >> 2] == kEvZero ? kEvFloor : ev[i >> 2];
                        if (wide & (1 << (i >> 2))) e = ev1[8 * (i >> 2) + (i & 3)];
                        sc[i] += e;
                        mx = fmaxf(mx, sc[i]);
                    }
                    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
                    for (int j = 0; j < 4; ++j) cj[j] = 1.0f, ev[j] = 0.0f;
                }
                const float m_new = mx > m_run + 8.0f ? __builtin_ceilf(mx) : m_run;
                const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[t][v] *= alpha;
                m_run = m_new;
            }
            const float off = m_run == -INFINITY ? 0.0f : -m_run;
            float pv[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float mo = ev[j] + off;
#pragma unroll
                for (int i = 4 * j; i < 4 * j + 4; ++i)
                    pv[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], cj[j], mo));
                l_run = __builtin_fmaf((pv[4 * j] + pv[4 * j + 1]) + (pv[4 * j + 2] + pv[4 * j + 3]), sm.vi[buf][j],
                                       l_run);
            }

            // ---- O^T += V^T P^T: step s takes the lane's weights i = 8s .. 8s + 7, keys 16s + 4p + 0..3
            // and 16s + 8 + 4p + 0..3; at head_dim 256 a block's terms are summed on their own first
            const int vrow = 4 * p + ((lane & 15) >> 2), vcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
            f16x8 ph[2], pl[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                f16x4 h0, l0, h1, l1;
                const float* w = pv + 8 * s;
                split4(w[0] * kPScale, w[1] * kPScale, w[2] * kPScale, w[3] * kPScale, h0, l0);
                split4(w[4] * kPScale, w[5] * kPScale, w[6] * kPScale, w[7] * kPScale, h1, l1);
                ph[s] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
                pl[s] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                f32x16 d;
#pragma unroll
                for (int v = 0; v < 16; ++v) d[v] = HD == 256 ? 0.0f : o[t][v];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    f16x8 f[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const f16x4 a0 = lds_transposed(&sm.v[buf][u][16 * s + vrow][32 * t + vcol]);
                        const f16x4 a1 = lds_transposed(&sm.v[buf][u][16 * s + 8 + vrow][32 * t + vcol]);
                        f[u] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                    }
                    d = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[1], ph[s], d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[0], pl[s], d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[0], ph[s], d, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) o[t][v] = HD == 256 ? o[t][v] + d[v] : d[v];
            }
        }
        if (!lead && more && __builtin_expect(commit_block(buf ^ 1), 0)) commit_wide(buf ^ 1, bi + G);
        __syncthreads();
    }
    l_run = (own_ref ? l_own : l_run) * kPScale;
    l_run += __shfl_xor(l_run, 32, 64);
    if (own_ref && l_run > 0.0f && l_run < INFINITY) {
        // o in the unit of l again: that of l's leading bit, in which o is no larger than a value
        const int k = __builtin_amdgcn_frexp_expf(l_run);
        const int eo = (int)__builtin_amdgcn_fmed3f(m_run - m_own - (float)k, -300.0f, 300.0f);
        l_run = __builtin_amdgcn_ldexpf(l_run, -k);
        m_run = m_own + (float)k;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[t][v] = __builtin_amdgcn_ldexpf(o[t][v], eo);
    }

    // ---- the second group's sums through LDS (its blocks are done with: the loop ends on a barrier)
    if constexpr (G == 2) {
        static_assert((16 * NT + 2) * 256 * sizeof(float) <= sizeof(smem), "");
        float* part = reinterpret_cast<float*>(smem) + tid;
        if (grp == 1) {
            part[0] = m_run, part[256] = l_run;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) part[256 * (2 + 16 * t + v)] = o[t][v];
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = part[0], m = fmaxf(m_run, m1);
        const float c0 = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m);
        const float c1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - m);
        m_run = m;
        l_run = l_run * c0 + part[256] * c1;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[t][v] = o[t][v] * c0 + part[256 * (2 + 16 * t + v)] * c1;
    }

    // ---- the lane's query row: dims 32t + 8(v/4) + 4p + v%4 of O^T / l, or with key splits
    // the unnormalised sums and (m, l) for the combine kernel (m = -inf, l = 0 if no key)
    if (q_ok) {
        if (a.splits == 1) {
            float* orow = a.out + (int64_t)tok * a.out_stride + (int64_t)h * HD;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) orow[32 * t + 8 * (v >> 2) + 4 * p + (v & 3)] = o[t][v] / l_run;
        } else {
            const int64_t wrow = ((int64_t)split * a.n_tokens + tok) * a.n_head + h;
            float* orow = a.ws_o + wrow * HD;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<float4*>(orow + 32 * t + 8 * j + 4 * p) =
                        make_float4(o[t][4 * j], o[t][4 * j + 1], o[t][4 * j + 2], o[t][4 * j + 3]);
            if (p == 0) {
                a.ws_ml[2 * wrow] = m_run;
                a.ws_ml[2 * wrow + 1] = l_run;
            }
        }
    }
}

hipError_t launch_attn_prompt(int ct, int hd, const AttnArgs& a, hipStream_t st) {
    const int64_t rows = (int64_t)a.n_tokens * (a.n_head / a.n_head_kv);
    const int64_t wgs = (rows + kRows - 1) / kRows * a.n_head_kv * a.splits;
    if (wgs > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs);
#define DCQ_PROMPT_CASE(C, H)                                                       \
    if (ct == C && hd == H) {                                                       \
        hipLaunchKernelGGL((attn_prompt_kernel<C, H>), grid, dim3(256 * prompt_groups(H)), 0, st, a); \
    } else
    DCQ_PROMPT_CASE(kTypeQ8_0, 128)
    DCQ_PROMPT_CASE(kTypeQ8_0, 64)
    DCQ_PROMPT_CASE(kTypeQ8_0, 256)
    DCQ_PROMPT_CASE(kTypeF16, 128)
    DCQ_PROMPT_CASE(kTypeF16, 64)
    DCQ_PROMPT_CASE(kTypeF16, 256)
    DCQ_PROMPT_CASE(kTypeF32, 128)
    DCQ_PROMPT_CASE(kTypeF32, 64)
    DCQ_PROMPT_CASE(kTypeF32, 256)
    return hipErrorNotSupported;
#undef DCQ_PROMPT_CASE
    return hipGetLastError();
}

}  // namespace dcq
