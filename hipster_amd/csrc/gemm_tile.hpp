// gemm_tile.hpp -- the prefill GEMM's tile kernel, D[m][n] = sum_k A[m][k] * bf16(W[n][k]), for every weight
// source of the call surface (Q4_K, Q5_K, IQ4_XS, Q6_K_SOA, Q8_0_SOA, Q5_1_SOA blocks and bf16 rows).
//
// A workgroup computes a tile of 32 NRB rows x 32 CW columns with CW x KS waves.  Wave (cw, kg) owns
// the 32 weight rows of column block cw and the K steps kg, kg + KS, ... of 64: it loads its rows'
// quantised bytes straight into registers, dequantises them into the MFMA operand (every weight
// once per row tile, no LDS round trip) and multiplies them with all NRB row blocks of A, which the CW
// waves of its K group share through a ring of ST LDS stages filled by DMA ST - 1 steps ahead.  The KS
// partial sums meet in LDS at the end, added in the order of kg (deterministic).
//
// Which k a lane holds is free as long as A and W agree: lane (r = l % 32, h = l / 32) of
// v_mfma_f32_32x32x16_bf16 supplies 8 values of its row per 16-wide slice, and the four slices of a
// step take them from the 16-byte run of quantised bytes that is contiguous in memory for that lane,
// so a step of 32 rows is one or two 16-byte loads per lane in every format.
//
// Measured against the 256 x 256 kernel it replaced, which dequantised through LDS and whose flat-form DMA made
// the compiler wait for every load in flight twice a step (HIP graph replay, weights rotated):
//   M x N x K              Q4_K             Q6_K
//   2048 x 17408 x 5120    429 -> 387 us    690 -> 539 us
//   2048 x 5120 x 17408    423 -> 354       704 -> 500
//   300 x 17408 x 5120     136 -> 74        210 -> 126
//   300 x 5120 x 17408     396 -> 93        683 -> 126
//   40 x 1024 x 5120       118 -> 11        191 -> 15
// What bounds it: with few rows the address units (a weight load touches 32 rows: about 80 cycles, A's DMA
// 1 KiB in 16-20), with many the matrix cores and the dequantisation beside them.
#pragma once
#include <type_traits>

#include "fmt_dequant.hpp"
#include "qmm_common.hpp"

namespace qmm {

constexpr int QMM_W_BF16 = 100;      // weight source: plain bf16 rows (not a wire format)

typedef __bf16 gt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gt_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 gt_h2 __attribute__((ext_vector_type(2)));

// The formats that pair a low and a high nibble of one byte run (Q4_K, Q5_K: sub-blocks 2j and 2j+1;
// Q6_K: quarters g and g + 2) give lane half h bytes 16h..16h+15 of the run: slices 0, 1 are the low
// nibbles, 2, 3 the high ones, and A's 16-byte chunk (8 values of k) of slice s is 4 (s / 2) + 2h + s % 2.
// The 32-weight formats (IQ4_XS, Q8_0, Q5_1) give lane half h the step's sub-block h: chunk 4h + s.
template <int F>
constexpr bool kHalfSub = F == QMM_IQ4_XS || F == QMM_Q8_0_SOA || F == QMM_Q5_1_SOA;
template <int F>
__device__ __forceinline__ int a_chunk(int s, int h) {
    if constexpr (kHalfSub<F>) return 4 * h + s;
    else return 4 * (s >> 1) + 2 * h + (s & 1);
}
// byte offset in an A row of step t, and of chunk c within the step.  A Q6_K step is quarters g and g+2 of
// a 128-weight half (the two nibbles of one ql run), so its chunks 4..7 lie 64 weights further on.
template <int F>
__device__ __forceinline__ uint32_t a_step_off(int t) {
    if constexpr (F == QMM_Q6_K_SOA) return (uint32_t)(t >> 1) * 256u + (uint32_t)(t & 1) * 64u;
    else return (uint32_t)t * 128u;
}
template <int F>
__device__ __forceinline__ uint32_t a_chunk_off(int c) {
    if constexpr (F == QMM_Q6_K_SOA) return (uint32_t)(16 * c + (c >= 4 ? 64 : 0));
    else return (uint32_t)(16 * c);
}

// a lane's quantised bytes of one step, loaded apart from their decode
template <int F>
struct WRaw {
    uint4 q;
    uint4 x;          // Q4_K, Q5_K: block header; Q8_0: second half of the sub-block; Q6_K: qh
    uint4 y;          // Q5_K: qh
    uint2 sc;         // scales: IQ4_XS header; Q6_K: the half's 8 scales; Q5_1: {qh, -}; Q8_0: {d, -}
    uint16_t d, m;    // Q6_K, Q8_0 d; Q5_1 d, m
};
template <>
struct WRaw<QMM_W_BF16> {
    uint4 v[4];
};

// buffer loads: rsrc covers the tile's rows, v the lane's byte offset in them, s the uniform one
typedef uint32_t gt_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t gt_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 bld16(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    const gt_u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
    return make_uint4(x.x, x.y, x.z, x.w);
}
__device__ __forceinline__ uint2 bld8(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    const gt_u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
    return make_uint2(x.x, x.y);
}
__device__ __forceinline__ uint32_t bld4(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0);
}
__device__ __forceinline__ uint16_t bld2(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, v, s, 0);
}

// w: the lane's row in the tile in bytes, h16 = 16 h, t the K step (uniform)
template <int F>
__device__ __forceinline__ void w_load(__amdgpu_buffer_rsrc_t b, uint32_t w, uint32_t h16, int K, uint32_t t, WRaw<F>& r) {
    if constexpr (F == QMM_W_BF16) {
        const uint32_t v = w + 2 * h16;
        r.v[0] = bld16(b, v, t * 128u);
        r.v[1] = bld16(b, v + 16, t * 128u);
        r.v[2] = bld16(b, v + 64, t * 128u);
        r.v[3] = bld16(b, v + 80, t * 128u);
    } else if constexpr (F == QMM_Q4_K) {
        r.x = bld16(b, w, (t >> 2) * 144u);
        r.q = bld16(b, w + h16, (t >> 2) * 144u + 16u + 32u * (t & 3));
    } else if constexpr (F == QMM_Q5_K) {
        r.x = bld16(b, w, (t >> 2) * 176u);
        r.y = bld16(b, w + h16, (t >> 2) * 176u + 16u);
        r.q = bld16(b, w + h16, (t >> 2) * 176u + 48u + 32u * (t & 3));
    } else if constexpr (F == QMM_IQ4_XS) {
        r.sc = bld8(b, w, (t >> 2) * 136u);
        r.q = bld16(b, w + h16, (t >> 2) * 136u + 8u + 32u * (t & 3));
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const uint32_t nb = (uint32_t)K >> 8, hf = t >> 1;                      // hf: 128-weight half of the row
        r.q = bld16(b, w + h16, 64u * hf + 32u * (t & 1));
        r.x = bld16(b, w + h16, nb * 128u + 32u * hf);
        r.sc = bld8(b, w, nb * 192u + 8u * hf);
        r.d = bld2(b, w, nb * 208u + 2u * (hf >> 1));
    } else if constexpr (F == QMM_Q8_0_SOA) {
        r.q = bld16(b, w + 2 * h16, 64u * t);
        r.x = bld16(b, w + 2 * h16 + 16, 64u * t);
        r.d = bld2(b, w + (h16 >> 3), (uint32_t)K + 4u * t);
    } else {                                                                       // QMM_Q5_1_SOA
        const uint32_t k8 = (uint32_t)K >> 3;
        r.q = bld16(b, w + h16, 32u * t);
        r.sc.x = bld4(b, w + (h16 >> 2), 4u * k8 + 8u * t);
        r.d = bld2(b, w + (h16 >> 3), 5u * k8 + 4u * t);
        r.m = bld2(b, w + (h16 >> 3), 5u * k8 + (k8 >> 1) + 4u * t);
    }
}

// every register of r is a use: the loads of this step have landed here
template <int F>
__device__ __forceinline__ void w_landed(const WRaw<F>& r) {
    if constexpr (F == QMM_W_BF16) {
        asm volatile("" ::"v"(r.v[0].x), "v"(r.v[1].x), "v"(r.v[2].x), "v"(r.v[3].x));
    } else if constexpr (F == QMM_Q4_K) {
        asm volatile("" ::"v"(r.q.x), "v"(r.x.x));
    } else if constexpr (F == QMM_Q5_K) {
        asm volatile("" ::"v"(r.q.x), "v"(r.x.x), "v"(r.y.x));
    } else if constexpr (F == QMM_IQ4_XS) {
        asm volatile("" ::"v"(r.q.x), "v"(r.sc.x));
    } else if constexpr (F == QMM_Q6_K_SOA) {
        asm volatile("" ::"v"(r.q.x), "v"(r.x.x), "v"(r.sc.x), "v"(r.d));
    } else if constexpr (F == QMM_Q8_0_SOA) {
        asm volatile("" ::"v"(r.q.x), "v"(r.x.x), "v"(r.d));
    } else {
        asm volatile("" ::"v"(r.q.x), "v"(r.sc.x), "v"(r.d), "v"(r.m));
    }
}

// the step's scales: w = fma(q, a, c) for slices 0, 1 and fma(q, a2, c2) for slices 2, 3 (q a small whole
// number held in an f16; where it is held as a subnormal, a carries the factor 2^24 or 2^20)
struct WScl { float a, c, a2, c2; };
template <int F>
__device__ __forceinline__ WScl w_scales(const WRaw<F>& r, int t, int h) {
    WScl o{0.f, 0.f, 0.f, 0.f};
    if constexpr (F == QMM_Q4_K || F == QMM_Q5_K) {
        const int j = t & 3;
        const float d = h2f(r.x.x), dmin = h2f(r.x.x >> 16);
        const Q4kScaleBytes sb = q4k_scale_bytes(r.x.y, r.x.z, r.x.w);
        o.a = d * (float)byte8(sb.sc_lo, sb.sc_hi, 2 * j) * 16777216.f;
        o.c = -(dmin * (float)byte8(sb.m_lo, sb.m_hi, 2 * j));
        o.a2 = d * (float)byte8(sb.sc_lo, sb.sc_hi, 2 * j + 1) * (F == QMM_Q4_K ? 1048576.f : 16777216.f);
        o.c2 = -(dmin * (float)byte8(sb.m_lo, sb.m_hi, 2 * j + 1));
    } else if constexpr (F == QMM_IQ4_XS) {
        const int ib = 2 * (t & 3) + h;
        const int ls = (int)((r.sc.y >> (4 * ib)) & 0xfu) | (int)(((r.sc.x >> (16 + 2 * ib)) & 3u) << 4);
        o.a = o.a2 = h2f(r.sc.x) * (float)(ls - 32);
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const int g = t & 1;
        const float d = h2f(r.d);
        o.a = d * (float)(int8_t)((r.sc.x >> (8 * (2 * g + h))) & 0xffu);
        o.a2 = d * (float)(int8_t)((r.sc.y >> (8 * (2 * g + h))) & 0xffu);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        o.a = o.a2 = h2f(r.d);
    } else if constexpr (F == QMM_Q5_1_SOA) {
        o.a = o.a2 = h2f(r.d) * 16777216.f;
        o.c = o.c2 = h2f(r.m);
    }
    return o;
}

// four unsigned bytes (0..31) -> bf16(fma(byte, s24 / 2^24, c)): the bytes as f16 subnormals
__device__ __forceinline__ void u4_bf16(uint32_t v, float s24, float c, gt_bf16x8& o, int i) {
    const uint32_t e = v & 0x00ff00ffu, d = (v >> 8) & 0x00ff00ffu;
    o[i] = (__bf16)mix_lo(e, s24, c);
    o[i + 1] = (__bf16)mix_lo(d, s24, c);
    o[i + 2] = (__bf16)mix_hi(e, s24, c);
    o[i + 3] = (__bf16)mix_hi(d, s24, c);
}
// four bytes b -> bf16(s * (b - bias)): b as the f16 number 1024 + b, exactly, minus 1024 + bias
__device__ __forceinline__ void s4_bf16(uint32_t v, float s, float bias, gt_bf16x8& o, int i) {
    const gt_h2 k = {(_Float16)(1024.f + bias), (_Float16)(1024.f + bias)};
    const uint32_t e = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gt_h2, (v & 0x00ff00ffu) | 0x64006400u) - k);
    const uint32_t d = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gt_h2, ((v >> 8) & 0x00ff00ffu) | 0x64006400u) - k);
    o[i] = (__bf16)mix_lo(e, s, 0.f);
    o[i + 1] = (__bf16)mix_lo(d, s, 0.f);
    o[i + 2] = (__bf16)mix_hi(e, s, 0.f);
    o[i + 3] = (__bf16)mix_hi(d, s, 0.f);
}

// slice s of the step: the lane's 8 weights, as qmm_dequant_bf16 gives them
template <int F>
__device__ __forceinline__ gt_bf16x8 w_slice(const WRaw<F>& r, const WScl& c, int t, int s) {
    gt_bf16x8 o;
    if constexpr (F == QMM_W_BF16) {
        o = __builtin_bit_cast(gt_bf16x8, r.v[s]);
    } else if constexpr (F == QMM_Q4_K) {
        const uint32_t u0 = s & 1 ? r.q.z : r.q.x, u1 = s & 1 ? r.q.w : r.q.y;
        o = s < 2 ? q4_bf16x8_mix(u0, u1, 0x000f000fu, c.a, c.c) : q4_bf16x8_mix(u0, u1, 0x00f000f0u, c.a2, c.c2);
    } else if constexpr (F == QMM_Q5_K) {
        const int bit = 2 * (t & 3) + (s >> 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t q = s & 1 ? (i ? r.q.w : r.q.z) : (i ? r.q.y : r.q.x);
            const uint32_t hb = s & 1 ? (i ? r.y.w : r.y.z) : (i ? r.y.y : r.y.x);
            const uint32_t v = ((s < 2 ? q : q >> 4) & 0x0f0f0f0fu) | (((hb >> bit) & 0x01010101u) << 4);
            u4_bf16(v, s < 2 ? c.a : c.a2, s < 2 ? c.c : c.c2, o, 4 * i);
        }
    } else if constexpr (F == QMM_IQ4_XS) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t q = s & 1 ? (i ? r.q.w : r.q.z) : (i ? r.q.y : r.q.x);
            // levels as unsigned bytes: signed level ^ 0x80 = level + 128
            s4_bf16(iq4_levels4((s < 2 ? q : q >> 4) & 0x0f0f0f0fu) ^ 0x80808080u, c.a, 128.f, o, 4 * i);
        }
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const int sh = 2 * ((t & 1) + (s < 2 ? 0 : 2));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t q = s & 1 ? (i ? r.q.w : r.q.z) : (i ? r.q.y : r.q.x);
            const uint32_t hb = s & 1 ? (i ? r.x.w : r.x.z) : (i ? r.x.y : r.x.x);
            const uint32_t v = ((s < 2 ? q : q >> 4) & 0x0f0f0f0fu) | (((hb >> sh) & 0x03030303u) << 4);
            s4_bf16(v, s < 2 ? c.a : c.a2, 32.f, o, 4 * i);
        }
    } else if constexpr (F == QMM_Q8_0_SOA) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint4 v = s < 2 ? r.q : r.x;
            s4_bf16((s & 1 ? (i ? v.w : v.z) : (i ? v.y : v.x)) ^ 0x80808080u, c.a, 128.f, o, 4 * i);
        }
    } else {                                            // QMM_Q5_1_SOA: slices 0, 1 weights 0..15 (low nibbles), 2, 3 weights 16..31
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t q = s & 1 ? (i ? r.q.w : r.q.z) : (i ? r.q.y : r.q.x);
            // bits 8s + 4i .. + 3 of qh, one per byte
            const uint32_t hb = ((((r.sc.x >> (8 * s + 4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u) << 4;
            u4_bf16(((s < 2 ? q : q >> 4) & 0x0f0f0f0fu) | hb, c.a, c.c, o, 4 * i);
        }
    }
    return o;
}

// Workgroup barrier over LDS while later stages' DMA stays in flight: this wave's LDS traffic is
// retired, the DMA a reader depends on has been waited for by its issuer before it
__device__ __forceinline__ void gt_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_s_waitcnt(0xC07F);       // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);
}

struct GemmArgs {
    const uint8_t* A;          // bf16 rows, lda bytes apart
    const uint8_t* W;          // weight rows, ldw bytes apart
    void* D;                   // f32 or bf16, rows ldd elements apart
    uint32_t lda, ldw, rowbytes;   // rowbytes: a weight row's own bytes
    int M, N, K, ldd;
};

// workgroup id -> tile: workgroup i runs on XCD i % 8, which takes a contiguous range of the tiles (M
// tiles fastest), so the M tiles that share weight rows share one L2
__device__ __forceinline__ void gt_tile(int bid, int ntiles, int mt, int& tm, int& tn) {
    const int x = bid & 7, q = ntiles >> 3, rem = ntiles & 7;
    const int id = x * q + (x < rem ? x : rem) + (bid >> 3);
    tm = id % mt;
    tn = id / mt;
}

template <int F, int NRB, int CW, int KS, int ST, bool OUT_BF16>
__device__ __forceinline__ void gemm_tile(const GemmArgs& a) {
    constexpr int BM = 32 * NRB, BN = 32 * CW, PF = ST - 1, NI = 4 * NRB, ND = (NI + CW - 1) / CW;
    constexpr int kStage = KS * BM * 8;                        // 16-byte slots per stage, all K groups
    static_assert(ST == 2 || ST == 4, "two or four stages");
    __shared__ uint4 s0[kStage], s1[kStage], s2[ST == 4 ? kStage : 1], s3[ST == 4 ? kStage : 1];
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    int tm, tn;
    gt_tile(blockIdx.x, mt * nt, mt, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63, fr = lane & 31, h = lane >> 5, fx = (fr >> 1) & 7;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cw = wave % CW, kg = wave / CW;
    const int nk = a.K >> 6, nit = (nk + KS - 1) / KS;
    // both operands through buffer resources over the tile's rows: their out-of-range offsets (rows past M
    // or N) read zeros without a memory access, and the DMA into LDS in this form leaves the compiler's count
    // of outstanding loads exact (the global form makes it wait for all of them)
    const int mrows = min(BM, a.M - m0), nrows = min(BN, a.N - n0);
    const uint8_t* const abase = a.A + (size_t)m0 * a.lda;
    const uint8_t* const wbase = a.W + (size_t)n0 * a.ldw;
    const int abytes = (int)((uint32_t)(mrows - 1) * a.lda + 2u * (uint32_t)a.K), wbytes = (int)((uint32_t)(nrows - 1) * a.ldw + a.rowbytes);
    const int ncol = 32 * cw + fr;
    const uint32_t woff = (uint32_t)ncol * a.ldw, h16 = 16u * (uint32_t)h;
    // DMA instruction q of the group's stage fills slots 64q + lane: rows 8q..8q+7, slot column lane % 8
    uint32_t aoff[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int q = min(cw + CW * i, NI - 1), r = 8 * q + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        aoff[i] = (uint32_t)r * a.lda + a_chunk_off<F>(c);
    }
    auto stage = [&](auto sc) -> uint4* {
        constexpr int S = decltype(sc)::value;
        if constexpr (S == 0) return s0;
        else if constexpr (S == 1) return s1;
        else if constexpr (S == 2) return s2;
        else return s3;
    };
    // K steps past the end read through an empty resource: zeros on both sides, no memory access
    auto issue = [&](auto sc, int it) {
        const int t = it * KS + kg;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)abase, 0, t < nk ? abytes : 0, 0x00020000);
        uint4* st = stage(sc) + kg * (BM * 8);
#pragma unroll
        for (int i = 0; i < ND; ++i)
            if (NI % CW == 0 || cw + CW * i < NI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(st + 64 * (cw + CW * i)), 16,
                                                         aoff[i], a_step_off<F>(t), 0, 0);
    };
    WRaw<F> raw[ST];
    auto wload = [&](int it, WRaw<F>& r) {
        const int t = it * KS + kg;
        w_load<F>(__builtin_amdgcn_make_buffer_rsrc((void*)wbase, 0, t < nk ? wbytes : 0, 0x00020000), woff, h16, a.K, (uint32_t)t, r);
    };
    auto frags = [&](auto sc, int s, gt_bf16x8 (&af)[NRB]) {
        const uint4* la = stage(sc) + kg * (BM * 8);
#pragma unroll
        for (int i = 0; i < NRB; ++i) {
            const uint4 v = la[(32 * i + fr) * 8 + (a_chunk<F>(s, h) ^ fx)];
            af[i] = __builtin_bit_cast(gt_bf16x8, v);
        }
    };
    gt_f32x16 acc[NRB];
#pragma unroll
    for (int i = 0; i < NRB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
    // prologue: steps 0 .. PF - 1 in flight
    issue(std::integral_constant<int, 0>(), 0);
    __builtin_amdgcn_sched_barrier(0);
    wload(0, raw[0]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ST == 4) {
        issue(std::integral_constant<int, 1>(), 1);
        __builtin_amdgcn_sched_barrier(0);
        wload(1, raw[1]);
        __builtin_amdgcn_sched_barrier(0);
        issue(std::integral_constant<int, 2>(), 2);
        __builtin_amdgcn_sched_barrier(0);
        wload(2, raw[2]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Loads land in order, so a step's weight bytes in registers mean that the A stage issued before them has
    // landed too.  With four stages the stage after the current one is complete at each barrier, so its
    // first fragments are read a step early.
    constexpr bool kAhead = ST == 4;
    w_landed<F>(raw[kAhead ? 1 : 0]);
    gt_barrier();
    WScl scl = w_scales<F>(raw[0], kg, h);
    gt_bf16x8 wv = w_slice<F>(raw[0], scl, kg, 0), af[NRB], afn[NRB];
    if constexpr (kAhead) frags(std::integral_constant<int, 0>(), 0, af);
    // step `it` in stage S: DMA and weight bytes of step it + PF go out first (into the stage that step it - 1
    // read), then the four slices' MFMAs, each beside the dequantisation of the slice after it
    auto body = [&](auto sc, int it) {
        constexpr int S = decltype(sc)::value, P = (S + PF) % ST, Nx = (S + 1) % ST;
        issue(std::integral_constant<int, P>(), it + PF);
        __builtin_amdgcn_sched_barrier(0);
        wload(it + PF, raw[P]);
        __builtin_amdgcn_sched_barrier(0);
        const int t = it * KS + kg, t1 = t + KS;
        if constexpr (!kAhead) frags(sc, 0, af);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) frags(sc, s + 1, afn);
            else if constexpr (kAhead) frags(std::integral_constant<int, Nx>(), 0, afn);
            gt_bf16x8 wn;
            if (s < 3) {
                wn = w_slice<F>(raw[S], scl, t, s + 1);
            } else {
                w_landed<F>(raw[Nx]);
                scl = w_scales<F>(raw[Nx], t1, h);
                wn = w_slice<F>(raw[Nx], scl, t1, 0);
            }
#pragma unroll
            for (int i = 0; i < NRB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], wv, acc[i], 0, 0, 0);
            constexpr int kV = (F == QMM_W_BF16 ? 0 : F == QMM_Q4_K ? 24 : 40) / NRB + 1;
#pragma unroll
            for (int i = 0; i < NRB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, kV, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            wv = wn;
#pragma unroll
            for (int i = 0; i < NRB; ++i) af[i] = afn[i];
        }
        w_landed<F>(raw[kAhead ? (S + 2) % ST : Nx]);
        gt_barrier();
    };
    int it = 0;
    for (; it + ST <= nit; it += ST) {
        body(std::integral_constant<int, 0>(), it);
        body(std::integral_constant<int, 1>(), it + 1);
        if constexpr (ST == 4) {
            body(std::integral_constant<int, 2>(), it + 2);
            body(std::integral_constant<int, 3>(), it + 3);
        }
    }
    if (it < nit) body(std::integral_constant<int, 0>(), it);
    if constexpr (ST == 4) {
        if (it + 1 < nit) body(std::integral_constant<int, 1>(), it + 1);
        if (it + 2 < nit) body(std::integral_constant<int, 2>(), it + 2);
    }
    __builtin_amdgcn_s_waitcnt(0);            // the clamped trailing DMAs
    auto put = [&](int i, int e, float v) {   // acc[i][e]: row 32i + 8(e/4) + 4h + e%4, column 32 cw + fr
        const int m = m0 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3), n = n0 + ncol;
        if (m < a.M && n < a.N) {
            if constexpr (OUT_BF16) ((uint16_t*)a.D)[(size_t)m * a.ldd + n] = (uint16_t)f2bf_bits(v);
            else ((float*)a.D)[(size_t)m * a.ldd + n] = v;
        }
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int i = 0; i < NRB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) put(i, e, acc[i][e]);
    } else {
        // partial sums through LDS (the ring is no longer needed): column block cw's KS partials, NRB x 16
        // x 64 floats each, fill stage cw; wave kg adds up and stores row-block registers kg, kg + KS, ...
        static_assert(KS * BM * 8 * 16 >= KS * NRB * 16 * 64 * 4, "a stage holds one column block's partial sums");
        static_assert(CW <= ST, "a stage per column block");
        __syncthreads();
        float* px = (float*)(cw == 0 ? s0 : cw == 1 ? s1 : cw == 2 ? s2 : s3);
#pragma unroll
        for (int i = 0; i < NRB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) px[((kg * NRB + i) * 16 + e) * 64 + lane] = acc[i][e];
        __syncthreads();
#pragma unroll
        for (int x = 0; x < NRB * 16 / KS; ++x) {
            const int ie = x * KS + kg, i = ie >> 4, e = ie & 15;
            float v = px[ie * 64 + lane];
#pragma unroll
            for (int g = 1; g < KS; ++g) v += px[(g * NRB * 16 + ie) * 64 + lane];
            put(i, e, v);
        }
    }
}

template <int F, int NRB, int CW, int KS, int ST, bool OUT_BF16>
__global__ void __launch_bounds__(64 * CW * KS) k_gemm_tile(GemmArgs a) {
    gemm_tile<F, NRB, CW, KS, ST, OUT_BF16>(a);
}

}  // namespace qmm
