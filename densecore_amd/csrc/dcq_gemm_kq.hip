// dcq_gemm_kq.hip — K-quant products (Q4_K, Q5_K, Q6_K) of many activation rows on gfx950 int8 MFMA, with
// the weight fragments built in registers.
//
// Replaces ggml's CPU MUL_MAT at M > 1 for K-quant weights (core/src/inference.cpp:1049-1063 and
// 1794-1797 route every M > 1 projection there; executed at core/src/worker.cpp:544), and the SwiGLU
// product of a gate/up pair (core/src/inference.cpp:1794-1796). Per activation row m, weight row n and
// superblock s (vec_dot_q4_K_q8_K and its siblings):
//   Y[m][n] = sum_s dA[m][s] * (d[n][s] * iS - dmin[n][s] * iM)
//   iS = sum over the 256 elements of qa * sc * q (Q6_K: sc * (q - 32)),  iM = sum_j m_j S_j (Q4_K, Q5_K)
// with iS and iM exact.
//
// Work split. A workgroup of 4 waves takes 32 MT activation rows x 128 weight rows; wave w owns weight
// rows 32 w .. 32 w + 31 and all the activation rows (MT MFMA tiles). K advances by superblocks, with the
// activation's 256 bytes per row double-buffered in LDS by direct-to-LDS loads (16-byte slots
// XOR-swizzled by the row) and shared by the four waves. A wave's weight rows are its own: lane (n, half)
// loads the bytes its MFMA operand needs straight from the superblock, one superblock ahead, and folds
// the sub-block scales into two int8 planes (64 registers) that then serve all MT tiles: no LDS traffic,
// no commit phase and one barrier per superblock.
//   Q4_K: q * sc = 8 q (sc >> 3) + q (sc & 7), both products at most 105.
//   Q5_K: the same planes reach 217, so they hold u - 128; the low plane's sums start from
//         1152 * (the row's sum of qa over the superblock), which the offsets of both planes come to.
//   Q6_K: w = sc (q - 32) is at most 4096 in magnitude: w = 256 hi + lo, lo in [-128, 127].
// The sums of a whole superblock stay in the MFMA's accumulators (v_mfma_i32_32x32x32_i8), so the VALU
// has one fp32 epilogue per 16 MFMAs. iM is one f16 MFMA per tile and superblock: the activation's
// 16-element sums are at most 2032 and the mins at most 63, both exact in f16, their products and sums
// exact in fp32.
// A SIMD issues one VALU instruction per 4 cycles at best (fma chains: 4.3 to 4.9 with two or four waves on
// it, 5.5 to 6.2 with one), an MFMA takes 32 cycles of its pipe: per tile and superblock 17 MFMAs are 544
// cycles and about 155 VALU instructions 620, where the kernel before had 31 VALU instructions per MFMA and
// its commit and barriers. Counters (2048 x 8192 x 2048, Q4_K): VALU busy 45 %, MFMA 35 %, a quarter of the
// MFMA time beside VALU, waits 38 %: neither unit is the limit, a wave's build, MFMAs and epilogue follow
// one another and two waves a SIMD overlap little of them.
//
// GLU: waves 0, 1 take 64 rows of the gate matrix and waves 2, 3 the same 64 of the up matrix; at the end
// the up waves pass their sums through LDS and the gate waves store silu(g) * u.
#include "dcq_common.h"
#include "dcq_kernels.h"

namespace dcq {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

enum { kQ4 = 0, kQ5 = 1, kQ6 = 2 };

// 16 (4) bytes per lane from global memory (uniform base + per-lane byte offset) into LDS at
// lds_base + 16 (4) * lane. Inline asm: the compiler's builtin form waits for every earlier LDS-direct
// load. Not counted by the compiler, so every call precedes the ordinary loads of its superblock (loads
// retire in order), and the superblock ends with an explicit s_waitcnt vmcnt(0) before the barrier.
__device__ __forceinline__ void dma16(const void* g, uint32_t off, const void* lds_base) {
    const uint32_t m0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds_base;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(g), "s"(m0) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void* g, uint32_t off, const void* lds_base) {
    const uint32_t m0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds_base;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(g), "s"(m0) : "memory", "m0");
}

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (v2us)(__builtin_bit_cast(v2us, a) * __builtin_bit_cast(v2us, b)));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(
        uint32_t, (v2us)(__builtin_bit_cast(v2us, a) * __builtin_bit_cast(v2us, b) + __builtin_bit_cast(v2us, c)));
}
// byte j of w in both halves of a dword
__device__ __forceinline__ uint32_t byte_pair(uint32_t w, int j) {
    return __builtin_amdgcn_perm(0u, w, 0x0c000c00u + 0x00010001u * (uint32_t)j);
}
// byte j of w as f16 in both halves
__device__ __forceinline__ uint32_t byte_half_pair(uint32_t w, int j) {
    const uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)(float)((w >> (8 * j)) & 0xFFu));
    return h * 0x00010001u;
}

// An empty use and redefinition: the value is in its registers here, for the compiler too.
__device__ __forceinline__ void pin(uint32_t& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(uint4& x) {
    v4i v = __builtin_bit_cast(v4i, x);
    asm volatile("" : "+v"(v));
    x = __builtin_bit_cast(uint4, v);
}

// One lane's weight bytes of a superblock, as loaded, and the operands built from them.
template <int F>
struct RawW;
template <>
struct RawW<kQ4> {
    uint4 hdr, qs[4];
    __device__ __forceinline__ void landed() {
        pin(hdr);
#pragma unroll
        for (int i = 0; i < 4; ++i) pin(qs[i]);
    }
    __device__ __forceinline__ void load(const uint8_t* b, int p) {
        hdr = ld16(b);
#pragma unroll
        for (int i = 0; i < 4; ++i) qs[i] = ld16(b + 16 + 32 * i + 16 * p);
    }
};
template <>
struct RawW<kQ5> {
    uint4 hdr, qh, qs[4];
    __device__ __forceinline__ void landed() {
        pin(hdr);
        pin(qh);
#pragma unroll
        for (int i = 0; i < 4; ++i) pin(qs[i]);
    }
    __device__ __forceinline__ void load(const uint8_t* b, int p) {
        hdr = ld16(b);
        qh = ld16(b + 16 + 16 * p);
#pragma unroll
        for (int i = 0; i < 4; ++i) qs[i] = ld16(b + 48 + 32 * i + 16 * p);
    }
};
template <>
struct RawW<kQ6> {
    uint32_t ql[4][4], qh[2][4], sc[4], d;  // blocks are 2-byte aligned
    __device__ __forceinline__ void landed() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j) pin(ql[i][j]);
            pin(qh[i >> 1][2 * (i & 1)]);
            pin(qh[i >> 1][2 * (i & 1) + 1]);
            pin(sc[i]);
        }
        pin(d);
    }
    __device__ __forceinline__ void load(const uint8_t* b, int p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_memcpy(ql[i], b + 32 * i + 16 * p, 16);
#pragma unroll
        for (int i = 0; i < 2; ++i) __builtin_memcpy(qh[i], b + 128 + 32 * i + 16 * p, 16);
        __builtin_memcpy(sc, b + 192, 16);
        d = ldu16(b + 208);
    }
};

struct FragW {
    v4i hi[8], lo[8];  // the planes' operands per sub-block of 32
    v8h mins;          // Q4_K, Q5_K: m of each 16-element group
    float d, dmin;
};

template <int F>
__device__ __forceinline__ void build(const RawW<F>& r, int p, FragW& f) {
    if constexpr (F == kQ6) {
        f.d = half_bits_to_float(r.d);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // sub-block j = quarter t of half h: lane half p holds its scale group 2 j + p
            const int h = j >> 2, t = j & 3;
            const uint32_t scw = r.sc[j >> 1] >> (8 * p);
            const uint32_t s16 = (uint32_t)__builtin_amdgcn_sbfe((int)scw, 16 * (j & 1), 8);
            const uint32_t s2 = __builtin_amdgcn_perm(s16, s16, 0x01000100u);
            const uint32_t c2 = pk_mad(s2, 0xFFE0FFE0u, 0x00800080u);  // 128 - 32 sc
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t nib = (r.ql[2 * h + (t & 1)][i] >> (t & 2 ? 4 : 0)) & 0x0F0F0F0Fu;
                const uint32_t q = nib | (((r.qh[h][i] >> (2 * t)) & 0x03030303u) << 4);
                const uint32_t we = pk_mad(q & 0x00FF00FFu, s2, c2), wo = pk_mad((q >> 8) & 0x00FF00FFu, s2, c2);
                f.hi[j][i] = (int)__builtin_amdgcn_perm(wo, we, 0x07030501u);
                f.lo[j][i] = (int)(__builtin_amdgcn_perm(wo, we, 0x06020400u) ^ 0x80808080u);
            }
        }
    } else {
        f.d = half_bits_to_float(r.hdr.x & 0xFFFF);
        f.dmin = half_bits_to_float(r.hdr.x >> 16);
        const uint32_t s0 = r.hdr.y, s1 = r.hdr.z, s2 = r.hdr.w;
        const uint32_t sc[2] = {s0 & 0x3F3F3F3Fu, (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)};
        const uint32_t m = p ? (((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) : s1 & 0x3F3F3F3Fu;
        v4i mm;  // groups 8 p + 0 .. 7 belong to sub-blocks 4 p + 0 .. 3
#pragma unroll
        for (int i = 0; i < 4; ++i) mm[i] = (int)byte_half_pair(m, i);
        f.mins = __builtin_bit_cast(v8h, mm);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t sh = byte_pair((sc[j >> 2] >> 3) & 0x07070707u, j & 3);
            const uint32_t sl = byte_pair(sc[j >> 2] & 0x07070707u, j & 3);
            const uint32_t w[4] = {r.qs[j >> 1].x, r.qs[j >> 1].y, r.qs[j >> 1].z, r.qs[j >> 1].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t q = (w[i] >> (j & 1 ? 4 : 0)) & 0x0F0F0F0Fu;
                if constexpr (F == kQ5) {
                    const uint32_t qh[4] = {r.qh.x, r.qh.y, r.qh.z, r.qh.w};
                    q |= ((qh[i] >> j) & 0x01010101u) << 4;
                }
                // byte products without carries: at most 15 * 7 (Q5_K: 31 * 7 = 217)
                const uint32_t x = F == kQ5 ? 0x80808080u : 0u;
                f.hi[j][i] = (int)(pk_mul(q, sh) ^ x);
                f.lo[j][i] = (int)(pk_mul(q, sl) ^ x);
            }
        }
    }
}

template <int F, int MT>
struct __align__(16) GemmSmem {
    uint8_t a[2][32 * MT * 256];
    float d[2][32 * MT < 64 ? 64 : 32 * MT];
    _Float16 s[2][F == kQ6 ? 1 : 32 * MT][16];      // the activation's 16-element sums
    int st[2][F == kQ5 ? 32 * MT : 4];              // 1152 * the superblock sum
};

constexpr int kXcds = 8;

}  // namespace

// W: K-quant rows (W2: the up matrix with GLU); xqs int8 [M][K], xd float [nsb][m_ld], xbs int16
// [M][K/16]. Y rows of y_stride floats, or the split's plane (splits > 1: plane s at Y + s * M * N,
// y_stride = N). R (optional): added to the result, row stride r_stride (0: one row).
//
// GRP: sums of grp superblocks are added to a second accumulator, so that the rounding of the running sum
// does not grow with K beyond the batch kernels' (they split K over eight waves). The products that come
// from those kernels take it, at one or two tiles a wave (what the LDS holds beside the staging).
template <int F, int MT, bool GLU, bool GRP>
__global__ void __launch_bounds__(256, MT == 1 ? 3 : 2) gemm_kq_kernel(const uint8_t* W, const uint8_t* W2, int64_t w_row_bytes, int N,
                                                         int nsb, const int8_t* xqs, const float* xd,
                                                         const int16_t* xbs, int m_ld, int M, int tiles_m, int tiles_n,
                                                         int stps, float* Y, int64_t y_stride, const float* R,
                                                         int64_t r_stride, int grp) {
    constexpr int BM = 32 * MT, BN = GLU ? 64 : 128;
    constexpr int BLOCK = F == kQ6 ? 210 : F == kQ5 ? 176 : 144;
    __shared__ GemmSmem<F, MT> sm;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int p = lane >> 5, c32 = lane & 31;
    const int tiles = tiles_m * tiles_n;
    const int split = blockIdx.x / tiles, bid = blockIdx.x - split * tiles;
    // XCD-aware tile order: XCD x (= id % 8) takes n-tile band x, walked m-first, so that a band's weight
    // rows stay in that XCD's L2
    int tile_m, tile_n;
    if (tiles_n % kXcds == 0) {
        const int band = tiles_n / kXcds, local = bid / kXcds;
        tile_n = bid % kXcds * band + local % band;
        tile_m = local / band;
    } else {
        tile_n = bid % tiles_n;
        tile_m = bid / tiles_n;
    }
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int64_t K = (int64_t)nsb * 256;
    const int sb0 = split * stps, sb1 = min(nsb, sb0 + stps);

    // ---- weights: the lane's row (clamped; rows past N are not stored)
    const uint8_t* wmat = GLU && wave >= 2 ? W2 : W;
    const int n = n0 + 32 * (GLU ? wave & 1 : wave) + c32;
    const uint8_t* wrow = wmat + (int64_t)min(n, N - 1) * w_row_bytes;
    RawW<F> raw;

    // ---- activation staging: wave w copies rows 4 w + 16 i .. + 3, 16 slots of 16 bytes each; slot k of row r
    // holds the row's piece k ^ (r & 15)
    uint32_t aoff[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int r = 16 * i + 4 * wave + (lane >> 4);
        aoff[i] = (uint32_t)((int64_t)min(r, M - 1 - m0) * K) + 16 * ((lane & 15) ^ (r & 15));
    }
    const int8_t* abase = xqs + (int64_t)m0 * K;
    // 16-element sums: thread -> row tid / 2, 8 of its 16
    const bool s_thread = F != kQ6 && tid < 2 * BM;
    const int16_t* sptr = F != kQ6 ? xbs + (int64_t)min(m0 + (tid >> 1), M - 1) * (K / 16) + 8 * (tid & 1) : nullptr;
    uint4 sraw = make_uint4(0, 0, 0, 0);

    auto issue = [&](int sb, int buf) {
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) dma16(abase + (int64_t)sb * 256, aoff[i], &sm.a[buf][(16 * i + 4 * wave) * 256]);
        if (wave < (MT + 1) / 2)  // m_ld covers whole 128-row tiles
            dma4(xd + (int64_t)sb * m_ld + m0 + 64 * wave, 4 * (MT == 1 ? lane & 31 : lane), &sm.d[buf][64 * wave]);
        if (F != kQ6 && s_thread) sraw = *reinterpret_cast<const uint4*>(sptr + (int64_t)sb * 16);
        raw.load(wrow + (int64_t)sb * BLOCK, p);
    };
    auto commit = [&](int buf) {
        if constexpr (F != kQ6) {
            const uint32_t w[4] = {sraw.x, sraw.y, sraw.z, sraw.w};
            v8h h;
            int sum = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int v = (int16_t)(w[i / 2] >> (16 * (i & 1)));
                h[i] = (_Float16)(short)v;
                sum += v;
            }
            if (s_thread) *reinterpret_cast<v8h*>(&sm.s[buf][tid >> 1][8 * (tid & 1)]) = h;
            if constexpr (F == kQ5) {
                sum += dpp_mov<0xB1>(sum);
                if (s_thread && (tid & 1) == 0) sm.st[buf][tid >> 1] = 1152 * sum;
            }
        }
    };

    v16f acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;

    // GRP: the groups' running total, the lane's own LDS words (registers would cost a wave per SIMD)
    __shared__ float tot[GRP ? 4 * 16 * MT * 64 : 1];
    float* mytot = tot + (GRP ? wave * 16 * MT * 64 + lane : 0);
    if constexpr (GRP) {
#pragma unroll
        for (int e = 0; e < 16 * MT; ++e) mytot[64 * e] = 0.0f;
    }

    issue(sb0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    raw.landed();
    commit(0);
    __syncthreads();
    for (int sb = sb0; sb < sb1; ++sb) {
        const int buf = (sb - sb0) & 1;
        FragW f;
        build<F>(raw, p, f);
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(f.hi[j]), "+v"(f.lo[j]));  // before the next loads
        if (sb + 1 < sb1) issue(sb + 1, buf ^ 1);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            v16i hi, lo;
            v16f mn;
#pragma unroll
            for (int i = 0; i < 16; ++i) hi[i] = 0, lo[i] = 0, mn[i] = 0.0f;
            if constexpr (F == kQ5) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const v4i s = *reinterpret_cast<const v4i*>(&sm.st[buf][32 * t + 8 * i + 4 * p]);
                    lo[4 * i] = s[0], lo[4 * i + 1] = s[1], lo[4 * i + 2] = s[2], lo[4 * i + 3] = s[3];
                }
            }
            const uint8_t* arow = &sm.a[buf][(32 * t + c32) * 256];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const v4i a = *reinterpret_cast<const v4i*>(arow + 16 * ((2 * j + p) ^ (c32 & 15)));
                hi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, f.hi[j], hi, 0, 0, 0);
                lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, f.lo[j], lo, 0, 0, 0);
            }
            if constexpr (F != kQ6)
                mn = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                    *reinterpret_cast<const v8h*>(&sm.s[buf][32 * t + c32][8 * p]), f.mins, mn, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 da = *reinterpret_cast<const float4*>(&sm.d[buf][32 * t + 8 * i + 4 * p]);
                const float dav[4] = {da.x, da.y, da.z, da.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int e = 4 * i + k;
                    // the fp32 steps of the kernels that dump block sums, so both give the same bits
                    const float is = (float)((int)((uint32_t)hi[e] << (F == kQ6 ? 8 : 3)) + lo[e]);
                    if constexpr (F == kQ6)
                        acc[t][e] = __builtin_fmaf(f.d * dav[k], is, acc[t][e]);
                    else
                        acc[t][e] = __builtin_fmaf(dav[k], __builtin_fmaf(-f.dmin, mn[e], f.d * is), acc[t][e]);
                }
            }
            asm volatile("" : "+v"(acc[t]));  // the epilogue stays here (it was sunk below every tile's MFMAs)
        }
        if constexpr (GRP) {
            if ((sb - sb0) % grp == grp - 1) {
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int i = 0; i < 16; ++i) mytot[64 * (16 * t + i)] += acc[t][i], acc[t][i] = 0.0f;
            }
        }
        // the next superblock's loads, issued before this one's MFMAs. landed(): without it the compiler
        // waits for them at their first use, behind the loads issued there after them
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        raw.landed();
        if (sb + 1 < sb1) commit(buf ^ 1);
        __syncthreads();
    }

    if constexpr (GRP) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][i] += mytot[64 * (16 * t + i)];
    }

    // ---- tile t, value i: row m0 + 32 t + 8 (i/4) + 4 p + i%4, column n
    if constexpr (GLU) {
        // the up waves' sums through the activation buffers (BM x 64 floats at most fill them)
        float* up = reinterpret_cast<float*>(sm.a[0]);
        if (wave >= 2) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) up[((wave & 1) * MT * 16 + t * 16 + i) * 64 + lane] = acc[t][i];
        }
        __syncthreads();
        if (wave >= 2) return;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][i] = silu(acc[t][i]) * up[(wave * MT * 16 + t * 16 + i) * 64 + lane];
    }
    if (n >= N) return;
    float* yp = Y + (int64_t)split * M * N + n;
    const float* rp = R ? R + n : nullptr;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = m0 + 32 * t + 8 * (i >> 2) + 4 * p + (i & 3);
            if (m < M) yp[(int64_t)m * y_stride] = rp ? acc[t][i] + rp[(int64_t)m * r_stride] : acc[t][i];
        }
}

typedef void (*GemmKqFn)(const uint8_t*, const uint8_t*, int64_t, int, int, const int8_t*, const float*, const int16_t*,
                         int, int, int, int, int, float*, int64_t, const float*, int64_t, int);

template <int F, bool GLU>
static GemmKqFn pick_mt(int mt, bool grp) {
    if (grp) return mt == 2 ? gemm_kq_kernel<F, 2, GLU, true> : gemm_kq_kernel<F, 1, GLU, true>;
    return mt == 4   ? gemm_kq_kernel<F, 4, GLU, false>
           : mt == 2 ? gemm_kq_kernel<F, 2, GLU, false>
                     : gemm_kq_kernel<F, 1, GLU, false>;
}

// Time of a CU's workgroups per superblock, us, when `load` of them fall to it: as many as its LDS and
// registers hold at once run together (two, or three at one tile a wave). Fitted to steps of 96 - 2048
// rows over six matrices (Q4_K, without grouped sums): e.g. 2560 x 9728 at 1024 rows, one tile a wave, 640
// workgroups: 2.6 x 38 superblocks = 98.8 us estimated and measured; four tiles 118 and 118.
static double gemm_us_per_sb(int wtype, int mt, int64_t load) {
    static const double c4[3] = {0.0, 3.1, 4.5}, c2[3] = {0.0, 1.9, 2.8}, c1[4] = {0.0, 1.2, 1.8, 2.6};
    const int64_t at_once = mt == 1 ? 3 : 2;
    const double* c = mt == 4 ? c4 : mt == 2 ? c2 : c1;
    // operands of Q5_K and Q6_K take more VALU work, which fewer tiles a wave share
    const double f = wtype == kTypeQ4_K ? 1.0 : wtype == kTypeQ5_K ? (mt == 4 ? 1.1 : mt == 2 ? 1.15 : 1.3)
                                                                    : (mt == 4 ? 1.25 : mt == 2 ? 1.5 : 2.0);
    return f * ((double)(load / at_once) * c[at_once] + c[load % at_once]);
}

struct GemmPlan {
    int mt, splits, stps;
};

// Tiles a wave (4, 2, 1) and K ranges with the least estimated time; a split adds the sum launch and its
// planes written and read at about 5 TB/s.
static GemmPlan plan_gemm(int wtype, int64_t M, int64_t N, int bn, int nsb, bool grp, const SplitScratch& sc) {
    const int64_t cus = cu_count(), plane = M * N * (int64_t)sizeof(float), tiles_n = (N + bn - 1) / bn;
    GemmPlan best{grp ? 2 : 4, 1, nsb};
    double best_us = 1e30;
    for (int mt = grp ? 2 : 4; mt >= 1; mt /= 2) {
        if (knob(Knob::GemmMt) > 0 && mt != knob(Knob::GemmMt)) continue;
        const int64_t tiles = (M + 32 * mt - 1) / (32 * mt) * tiles_n;
        for (int s = 1; s <= 8 && (s == 1 || (sc.p && nsb / s >= 4 && (size_t)(s * plane) <= sc.bytes)); ++s) {
            const int stps = (nsb + s - 1) / s, splits = (nsb + stps - 1) / stps;
            double us = gemm_us_per_sb(wtype, mt, (tiles * splits + cus - 1) / cus) * stps;
            if (splits > 1) us += 2.0 + 2.0 * splits * (double)plane / 5.0e6;
            if (us < best_us) best_us = us, best = GemmPlan{mt, splits, stps};
        }
    }
    return best;
}

// Steps (us) on the kernels that serve these products otherwise -> on this one, MI355X, 5 - 2048 rows over 14
// matrices. Plain products:
//   Q4_K, Q5_K: from 513 rows always (768 x 4096 x 4096 72.5 -> 50.9, 2048 x 9728 x 2560 155 -> 136, 520 x 256 x
//     2560 18.8 -> 14.9; Q5_K 79.0 -> 62.4, 163 -> 156, 19.2 -> 18.0). From 65 rows by M N: 200 x 8192 x 2048 27.5 ->
//     23.9, 384 x 5120 x 2560 31.2 -> 28.0 (Q5_K 31.2 -> 28.1, 35.3 -> 32.4), but 384 x 4096 x 4096 33.3 against
//     34.8; tall ones earlier, 160 x 9728 x 2560 30.3 -> 26.5, 96 x 28672 x 4096 68.5 -> 47.9, but Q5_K 128 x 9728 x
//     2560 27.1 against 29.0
//   Q6_K from 65 rows: where 128 x 128 tiles are more than the CUs, which the prefill kernel serves one at a
//     time: 129 x 16400 x 2048 63.0 -> 43.7, 600 x 9728 x 2560 76.0 -> 66.8, but 512 x 8192 x 2048 35.5 against 38.7
//   33 - 64 rows over 25600 weight rows or more: 64 x 25600 x 2560 29.3 -> 25.5, Q5_K 34.0 -> 30.9, Q6_K 48 x 28672
//     x 4096 66.4 -> 59.0; but 48 x 14336 x 4096 22.7 against 24.7
//   fewer, under 8 superblocks (the batch kernels' waves split K eight ways) on tall matrices: 16 x 151936 x
//     1024 49.8 -> 28.4, Q5_K 59.2 -> 42.4, Q6_K 75.9 -> 49.3; 16 x 32768 x 1792 17.8 -> 16.4, but Q5_K 20.3 against
//     21.4
//   Q6_K rows of an odd number of superblocks, which only the generic kernel takes: 1000 x 9728 x 2816 469 -> 119,
//     64 x 2560 x 9472 111 -> 30.0, 33 x 1024 x 1280 22.2 -> 18.5; but 16 x 4096 x 2816 21.5 against 24.8, 33 x 1024 x
//     1792 24.2 against 26.3, and without room to split K (the generic kernel's waves split it) 5 x 2048 x 11008 54
//     against 138, 192 x 2048 x 7936 77 against 102, while 192 x 4096 x 7936 102 and 103, 512 x 4096 x 7936 222 -> 109
// Gate/up pairs (against two products and the SiLU kernel):
//   Q4_K, Q5_K: 2048 x 9728 x 2560 345 -> 279 (Q5_K 355 -> 321), 256 x 4096 x 4096 48.1 -> 41.0, 72 x 8192 x 2048
//     30.7 -> 22.2, 16 x 9728 x 2560 21.9 -> 19.1; but 128 x 4096 x 4096 27.1 against 28.9, 64 x 4096 x 4096 20.3
//     against 27.9, Q5_K 16 x 9728 x 2560 25.1 against 26.0
//   Q6_K: 2048 x 9728 x 2560 396 -> 318, 72 x 8192 x 2048 35.5 -> 30.0, 512 x 1024 x 2560 41.7 -> 30.8, 48 x 9728 x
//     2560 48.6 -> 36.4; but 128 x 4096 x 4096 37.3 against 47.7, 32 x 9728 x 2560 31.3 against 31.6
//   Long rows of few tiles, where the two products split K and the pair cannot: Q6_K 512 x 1024 x 13824 78 against
//     143, 1200 x 1024 x 6144 86 against 107, 160 tiles x 16 superblocks 69 against 76, but 1200 x 2048 x 6144 177 -> 148,
//     256 x 4096 x 4096 58 -> 54; Q5_K 600 x 256 x 6144 50 against 57, 1200 x 512 x 13824 117 against 133; Q4_K 600 x
//     256 x 13824 63 against 75
bool gemm_kq_wins(int wtype, int64_t M, int64_t N, int64_t K, bool glu, const SplitScratch& sc) {
    if ((wtype != kTypeQ4_K && wtype != kTypeQ5_K && wtype != kTypeQ6_K) || M <= 4) return false;
    if (knob(Knob::GemmKq) >= 0) return knob(Knob::GemmKq) != 0;
    const int64_t nsb = K / 256;
    if (wtype == kTypeQ6_K && nsb % 2) {
        const bool split = !glu && nsb >= 8 && sc.p && sc.bytes >= (size_t)(2 * M * N) * sizeof(float);
        if (M <= 32) return split && nsb >= 11 && N * K >= (int64_t)1 << (nsb >= 13 ? 24 : 25);
        if (glu || nsb <= 5 || (M <= 64 && N >= 16384 && nsb <= 16)) return true;
        if (split && (nsb >= 11 || M > 48)) return true;
        return M * N >= (nsb <= 16 ? 600000 : 800000);
    }
    if (glu) {
        if (wtype == kTypeQ6_K) {
            const int64_t tiles = (M + 127) / 128 * ((N + 63) / 64);
            if (M <= 32 || tiles < (M > 256 ? 64 : 128)) return false;
            return M <= 64 || nsb <= 12 || tiles >= 192 || (nsb <= 16 && tiles >= 96 && tiles <= 128);
        }
        if (M <= 64) return N >= 9216 && (M > 32 || wtype == kTypeQ4_K);
        if (M > 512) return wtype == kTypeQ4_K ? nsb <= 24 || M * N >= 250000 : nsb <= 16 || M * N >= 700000;
        return N >= 8192 || M * N >= 1000000;
    }
    if (M <= 32) return nsb < 8 && N >= (wtype == kTypeQ5_K ? 65536 : 32768);
    if (M <= 64) return N >= 25600;
    if (wtype == kTypeQ6_K) return ((M + 127) / 128) * ((N + 127) / 128) > (int64_t)cu_count();
    return M > 512 || M * N >= (N >= 9216 ? 1300000 : 1600000);
}

hipError_t launch_gemm_kq(int wtype, const void* W, const void* W2, int64_t w_row_bytes, int64_t N, int64_t K,
                          const PlanarBuffers& act, int64_t M, float* Y, int64_t y_stride, hipStream_t st,
                          const SplitScratch& sc) {
    const int64_t nsb = K / 256;
    if (K % 256 || nsb < 1 || N > INT32_MAX || M > INT32_MAX || K > ((int64_t)1 << 24) || act.m_ld % 128)
        return hipErrorNotSupported;
    const bool glu = W2 != nullptr;
    const int bn = glu ? 64 : 128;
    // grouped sums where a kernel that splits K over its waves would serve the product (the batch kernels, the
    // generic one below 512 of its tiles); the 128 x 128-tile kernels add superblocks one by one, as without
    const bool q6 = wtype == kTypeQ6_K;
    const int64_t tiles128 = (M + 127) / 128 * ((N + 127) / 128);
    const bool grp = M <= 64 || (q6 ? nsb % 2 && (M + 63) / 64 * ((N + 255) / 256) < 512
                                    : M <= 256 || (M <= 512 && tiles128 < (int64_t)cu_count()));
    const GemmPlan pl = plan_gemm(wtype, M, N, bn, (int)nsb, grp, glu ? SplitScratch() : sc);
    const int64_t tiles_n = (N + bn - 1) / bn, tiles_m = (M + 32 * pl.mt - 1) / (32 * pl.mt);
    if (tiles_m * tiles_n * pl.splits > INT32_MAX) return hipErrorNotSupported;
    const GemmKqFn fn = wtype == kTypeQ4_K   ? (glu ? pick_mt<kQ4, true>(pl.mt, grp) : pick_mt<kQ4, false>(pl.mt, grp))
                        : wtype == kTypeQ5_K ? (glu ? pick_mt<kQ5, true>(pl.mt, grp) : pick_mt<kQ5, false>(pl.mt, grp))
                                             : (glu ? pick_mt<kQ6, true>(pl.mt, grp) : pick_mt<kQ6, false>(pl.mt, grp));
    float* out = pl.splits > 1 ? sc.p : Y;
    int64_t out_stride = pl.splits > 1 ? N : y_stride, r_stride = 0;
    const float* R = nullptr;
    if (sc.add && pl.splits == 1 && !glu) {
        R = sc.add->R, r_stride = sc.add->r_stride, out = sc.add->Y, out_stride = sc.add->y_stride;
        sc.add->done = true;
    }
    int group = 2;  // about the root of the superblocks: as many roundings within a group as across them
    while ((group + 1) * (group + 1) <= pl.stps) ++group;
    hipLaunchKernelGGL(fn, dim3((unsigned)(tiles_m * tiles_n * pl.splits)), dim3(256), 0, st, (const uint8_t*)W,
                       (const uint8_t*)W2, w_row_bytes, (int)N, (int)nsb, act.qs, act.d, act.bs, (int)act.m_ld, (int)M,
                       (int)tiles_m, (int)tiles_n, pl.stps, out, out_stride, R, r_stride, group);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || pl.splits == 1) return e;
    return launch_sum_splits(sc, pl.splits, M, N, Y, y_stride, st);
}

}  // namespace dcq
