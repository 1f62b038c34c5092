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
//   2048 x 17408 x 5120    429 -> 385 us    690 -> 437 us
//   2048 x 5120 x 17408    423 -> 346       704 -> 397
//   300 x 17408 x 5120     136 -> 72        210 -> 90
//   300 x 5120 x 17408     396 -> 94        683 -> 121
//   40 x 1024 x 5120       118 -> 9.6       191 -> 12.6
// What bounds it.  With many rows the card's power: the matrix cores are 60% busy at 1.7 GHz (Q4_K, 192 x 256
// tiles), about what a library bf16 product of that size reaches.  With few rows the vector memory path: a load of
// one row per lane costs the address units 50-80 cycles whatever its width, and without the weight loads
// 300 x 17408 x 5120 took 53 us instead of 73 (no dequantisation 62, no matrix instructions 59, eight
// stages instead of four the same).  Hence the scales and high bits of four steps in one load (a step's loads
// Q4_K 2 -> 1.25, Q5_K 3 -> 1.5, Q6_K 4 -> 2, Q5_1 4 -> 2; Q6_K at 2048 x 17408 x 5120 494 -> 398 us) and the loads of
// a step spread over its slices.  Measured and not kept: the weight rows through LDS by DMA with consecutive lanes on
// consecutive bytes (the same times: the LDS traffic and the waits took back what the address units gained), six
// and eight stages, two to four smaller workgroups per CU.
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

// A lane's weights of one step: its quants, loaded every step (WQ), and the block's scales and high bits, loaded
// once per chunk of CK steps (WHead) and decoded for all of them at once (WDec): a load of one row per lane costs
// the address units 50-80 cycles whatever its width, and a scale byte at a fixed place decodes in one
// instruction.
template <int F>
struct WQ {
    uint4 q;
    uint4 x;          // Q8_0: second half of the sub-block
};
template <>
struct WQ<QMM_W_BF16> {
    uint4 v[4];
};
template <int F>
struct WHead {
    uint4 x;          // Q4_K, Q5_K: block header; Q6_K: scales; Q8_0, Q5_1: d
    uint4 y[2];       // Q5_K: qh of the lane half; Q6_K: qh of the chunk's halves; Q5_1: qh
    uint4 m;          // Q5_1: m
    uint2 sc;         // IQ4_XS: block header
    uint16_t d;       // Q6_K: d
};
// weights of step u of the chunk: fma(q, a[u], c[u]) in slices 0, 1 and fma(q, a2[u], c2[u]) in slices 2, 3 (q a
// whole number in an f16; where it is held as a subnormal, a carries the factor 2^24 or 2^20); the formats of one
// scale per lane and step use a and c only
template <int F, int CK>
struct WDec {
    float a[CK], c[CK], a2[CK], c2[CK];
    uint4 hi[CK / 2];         // Q5_K: qh in hi[0]; Q6_K: qh of the halves
    uint32_t qh[CK];          // Q5_1
};

// w: the lane's row in the tile in bytes, h16 = 16 h, t the K step (uniform)
template <int F>
__device__ __forceinline__ void wq_load(__amdgpu_buffer_rsrc_t b, uint32_t w, uint32_t h16, uint32_t t, WQ<F>& r) {
    if constexpr (F == QMM_W_BF16) {
        const uint32_t v = w + 2 * h16;
        r.v[0] = bld16(b, v, t * 128u);
        r.v[1] = bld16(b, v + 16, t * 128u);
        r.v[2] = bld16(b, v + 64, t * 128u);
        r.v[3] = bld16(b, v + 80, t * 128u);
    } else if constexpr (F == QMM_Q4_K) {
        r.q = bld16(b, w + h16, (t >> 2) * 144u + 16u + 32u * (t & 3));
    } else if constexpr (F == QMM_Q5_K) {
        r.q = bld16(b, w + h16, (t >> 2) * 176u + 48u + 32u * (t & 3));
    } else if constexpr (F == QMM_IQ4_XS) {
        r.q = bld16(b, w + h16, (t >> 2) * 136u + 8u + 32u * (t & 3));
    } else if constexpr (F == QMM_Q6_K_SOA) {
        r.q = bld16(b, w + h16, 32u * t);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        r.q = bld16(b, w + 2 * h16, 64u * t);
        r.x = bld16(b, w + 2 * h16 + 16, 64u * t);
    } else {
        r.q = bld16(b, w + h16, 32u * t);
    }
}
// t0: the chunk's first step, a multiple of CK (2 or 4)
template <int F, int CK>
__device__ __forceinline__ void wh_load(__amdgpu_buffer_rsrc_t b, uint32_t w, uint32_t h16, int K, uint32_t t0, WHead<F>& r) {
    const uint32_t nb = (uint32_t)K >> 8, k8 = (uint32_t)K >> 3;
    if constexpr (F == QMM_Q4_K) {
        r.x = bld16(b, w, (t0 >> 2) * 144u);
    } else if constexpr (F == QMM_Q5_K) {
        r.x = bld16(b, w, (t0 >> 2) * 176u);
        r.y[0] = bld16(b, w + h16, (t0 >> 2) * 176u + 16u);
    } else if constexpr (F == QMM_IQ4_XS) {
        r.sc = bld8(b, w, (t0 >> 2) * 136u);
    } else if constexpr (F == QMM_Q6_K_SOA) {
        if constexpr (CK == 4) r.x = bld16(b, w, nb * 192u + 4u * t0);
        else r.sc = bld8(b, w, nb * 192u + 4u * t0);
        r.y[0] = bld16(b, w + h16, nb * 128u + 16u * t0);
        if constexpr (CK == 4) r.y[1] = bld16(b, w + h16, nb * 128u + 16u * t0 + 32u);
        r.d = bld2(b, w, nb * 208u + 2u * (t0 >> 2));
    } else if constexpr (F == QMM_Q8_0_SOA) {
        if constexpr (CK == 4) r.x = bld16(b, w, (uint32_t)K + 4u * t0);
        else r.sc = bld8(b, w, (uint32_t)K + 4u * t0);
    } else if constexpr (F == QMM_Q5_1_SOA) {
        r.y[0] = bld16(b, w, 4u * k8 + 8u * t0);
        if constexpr (CK == 4) {
            r.y[1] = bld16(b, w, 4u * k8 + 8u * t0 + 16u);
            r.x = bld16(b, w, 5u * k8 + 4u * t0);
            r.m = bld16(b, w, 5u * k8 + (k8 >> 1) + 4u * t0);
        } else {
            const uint2 d = bld8(b, w, 5u * k8 + 4u * t0), m = bld8(b, w, 5u * k8 + (k8 >> 1) + 4u * t0);
            r.sc = d;
            r.m.x = m.x;
            r.m.y = m.y;
        }
    }
}

// a use of a step's quants: its loads have landed here
template <int F>
__device__ __forceinline__ void wq_landed(const WQ<F>& r) {
    if constexpr (F == QMM_W_BF16) asm volatile("" ::"v"(r.v[0].x), "v"(r.v[1].x), "v"(r.v[2].x), "v"(r.v[3].x));
    else if constexpr (F == QMM_Q8_0_SOA) asm volatile("" ::"v"(r.q.x), "v"(r.x.x));
    else asm volatile("" ::"v"(r.q.x));
}

// byte i of word w as a float (i known at compile time: one instruction)
__device__ __forceinline__ float ub(uint32_t w, int i) { return (float)((w >> (8 * i)) & 0xffu); }
__device__ __forceinline__ uint32_t word(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// t0 as in wh_load; steps from nk on belong to no weight (their bytes are other data): scale 0
template <int F, int CK>
__device__ __forceinline__ void wh_decode(const WHead<F>& r, int t0, int nk, int h, WDec<F, CK>& o) {
    if constexpr (F == QMM_Q4_K || F == QMM_Q5_K) {
        const float d = h2f(r.x.x), dmin = h2f(r.x.x >> 16);
        const float d24 = d * 16777216.f, dhi = d * (F == QMM_Q4_K ? 1048576.f : 16777216.f), nm = -dmin;
        const Q4kScaleBytes sb = q4k_scale_bytes(r.x.y, r.x.z, r.x.w);
        const bool up = CK == 2 && (t0 & 2);
        const uint32_t s0 = up ? sb.sc_hi : sb.sc_lo, m0 = up ? sb.m_hi : sb.m_lo;
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t s = u < 2 ? s0 : sb.sc_hi, m = u < 2 ? m0 : sb.m_hi;
            o.a[u] = d24 * ub(s, 2 * (u & 1));
            o.c[u] = nm * ub(m, 2 * (u & 1));
            o.a2[u] = dhi * ub(s, 2 * (u & 1) + 1);
            o.c2[u] = nm * ub(m, 2 * (u & 1) + 1);
        }
        if constexpr (F == QMM_Q5_K) o.hi[0] = r.y[0];
    } else if constexpr (F == QMM_IQ4_XS) {
        const float d = h2f(r.sc.x);
        const uint32_t sl = r.sc.y >> (4 * h + (CK == 2 ? 8 * (t0 & 3) : 0)), sh = r.sc.x >> (16 + 2 * h + (CK == 2 ? 4 * (t0 & 3) : 0));
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const int ls = (int)((sl >> (8 * u)) & 0xfu) | (int)(((sh >> (4 * u)) & 3u) << 4);
            o.a[u] = d * (float)(ls - 32);
        }
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const float d = h2f(r.d);
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t s0 = CK == 2 ? r.sc.x : word(r.x, u & 2), s1 = CK == 2 ? r.sc.y : word(r.x, (u & 2) + 1);
            o.a[u] = d * (float)(int8_t)((s0 >> (8 * h)) >> (16 * (u & 1)));
            o.a2[u] = d * (float)(int8_t)((s1 >> (8 * h)) >> (16 * (u & 1)));
        }
#pragma unroll
        for (int v = 0; v < CK / 2; ++v) o.hi[v] = r.y[v];
    } else if constexpr (F == QMM_Q8_0_SOA) {
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t v = CK == 2 ? (u ? r.sc.y : r.sc.x) : word(r.x, u);
            o.a[u] = t0 + u < nk ? h2f(v >> (16 * h)) : 0.f;
        }
    } else if constexpr (F == QMM_Q5_1_SOA) {
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t v = CK == 2 ? (u ? r.sc.y : r.sc.x) : word(r.x, u), m = word(r.m, u);
            o.a[u] = t0 + u < nk ? h2f(v >> (16 * h)) * 16777216.f : 0.f;
            o.c[u] = t0 + u < nk ? h2f(m >> (16 * h)) : 0.f;
            const uint4 y = r.y[u >> 1];
            o.qh[u] = u & 1 ? (h ? y.w : y.z) : (h ? y.y : y.x);
        }
    }
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

// slice s of step u of the chunk (step t): the lane's 8 weights, as qmm_dequant_bf16 gives them
template <int F, int CK>
__device__ __forceinline__ gt_bf16x8 w_slice(const WQ<F>& r, const WDec<F, CK>& c, int t, int u, int s) {
    gt_bf16x8 o;
    if constexpr (F == QMM_W_BF16) {
        o = __builtin_bit_cast(gt_bf16x8, r.v[s]);
    } else if constexpr (F == QMM_Q4_K) {
        const uint32_t u0 = s & 1 ? r.q.z : r.q.x, u1 = s & 1 ? r.q.w : r.q.y;
        o = s < 2 ? q4_bf16x8_mix(u0, u1, 0x000f000fu, c.a[u], c.c[u]) : q4_bf16x8_mix(u0, u1, 0x00f000f0u, c.a2[u], c.c2[u]);
    } else {
        // chunks of four steps start at a multiple of four, so the step within the block is known at compile time
        const int j = CK == 4 ? u : (t & 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int w = 2 * (s & 1) + i;
            const uint32_t q = word(r.q, w), nib = (s < 2 ? q : q >> 4) & 0x0f0f0f0fu;
            if constexpr (F == QMM_Q5_K) {
                const uint32_t v = nib | (((word(c.hi[0], w) >> (2 * j + (s >> 1))) & 0x01010101u) << 4);
                u4_bf16(v, s < 2 ? c.a[u] : c.a2[u], s < 2 ? c.c[u] : c.c2[u], o, 4 * i);
            } else if constexpr (F == QMM_IQ4_XS) {      // levels as unsigned bytes: signed level ^ 0x80 = level + 128
                s4_bf16(iq4_levels4(nib) ^ 0x80808080u, c.a[u], 128.f, o, 4 * i);
            } else if constexpr (F == QMM_Q6_K_SOA) {
                const uint32_t v = nib | (((word(c.hi[u >> 1], w) >> (2 * (u & 1) + (s < 2 ? 0 : 4))) & 0x03030303u) << 4);
                s4_bf16(v, s < 2 ? c.a[u] : c.a2[u], 32.f, o, 4 * i);
            } else if constexpr (F == QMM_Q8_0_SOA) {
                s4_bf16((s < 2 ? q : word(r.x, w)) ^ 0x80808080u, c.a[u], 128.f, o, 4 * i);
            } else {                                     // QMM_Q5_1_SOA: bits 8s + 4i .. + 3 of qh, one per byte
                const uint32_t hb = ((((c.qh[u] >> (8 * s + 4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u) << 4;
                u4_bf16(nib | hb, c.a[u], c.c[u], o, 4 * i);
            }
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

// steps of a chunk, and the steps that every K group runs for nk steps of 64
__host__ __device__ constexpr int gt_chunk(int ks) { return ks == 8 ? 2 : 4; }
__host__ __device__ constexpr int gt_local_steps(int nk, int ks) {
    const int ck = gt_chunk(ks), nch = (nk + ck - 1) / ck;
    return ks == 1 ? nk : ck * ((nch + ks - 1) / ks);
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

// One tile.  s0..s3: the ring's stages (s2, s3 unused when ST = 2), at least KS * 32 NRB * 8 slots each and
// separate __shared__ arrays: the compiler then knows which stage a DMA writes and an LDS read waits for
// that stage only.  abase / wbase: the operands' tile, abytes / wbytes its extent; arow(r): byte offset of A's
// row r in it; put(i, e, v): register e of row block i, which is row 32i + 8(e/4) + 4h + e%4, column 32 cw + fr.
template <int F, int NRB, int CW, int KS, int ST, class ARow, class Put>
__device__ __forceinline__ void gemm_tile_core(uint4* s0, uint4* s1, uint4* s2, uint4* s3, const uint8_t* abase, uint32_t abytes,
                                               const uint8_t* wbase, uint32_t wbytes, uint32_t ldw, int K, const ARow& arow,
                                               const Put& put) {
    constexpr int BM = 32 * NRB, PF = ST - 1, NI = 4 * NRB, ND = (NI + CW - 1) / CW;
    static_assert(ST == 2 || ST == 4, "two or four stages");
    const int lane = threadIdx.x & 63, fr = lane & 31, h = lane >> 5, fx = (fr >> 1) & 7;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cw = wave % CW, kg = wave / CW;
    // K groups take chunks of CK steps in turn; local step it of group kg is step kstep(it)
    constexpr int CK = gt_chunk(KS);
    const int nk = K >> 6, nit = gt_local_steps(nk, KS);
    auto kstep = [&](int it) { return KS == 1 ? it : ((int)((unsigned)it / CK) * KS + kg) * CK + (int)((unsigned)it % CK); };
    const uint32_t woff = (uint32_t)(32 * cw + fr) * ldw, h16 = 16u * (uint32_t)h;
    // DMA instruction q of the group's stage fills slots 64q + lane: rows 8q..8q+7, slot column lane % 8
    uint32_t aoff[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int q = min(cw + CW * i, NI - 1), r = 8 * q + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        aoff[i] = arow(r) + a_chunk_off<F>(c);
    }
    auto stage = [&](auto sc) -> uint4* {
        constexpr int S = decltype(sc)::value;
        if constexpr (S == 0) return s0;
        else if constexpr (S == 1) return s1;
        else if constexpr (S == 2) return s2;
        else return s3;
    };
    // K steps past the end read through an empty resource: zeros on both sides, no memory access
    auto issue = [&](auto sc, int it, int i0, int i1) {
        const int t = kstep(it);
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)abase, 0, t < nk ? (int)abytes : 0, 0x00020000);
        uint4* st = stage(sc) + kg * (BM * 8);
#pragma unroll
        for (int i = 0; i < ND; ++i)
            if (i >= i0 && i < i1 && (NI % CW == 0 || cw + CW * i < NI))
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(st + 64 * (cw + CW * i)), 16,
                                                         aoff[i], a_step_off<F>(t), 0, 0);
    };
    WQ<F> raw[ST];
    // the head of a chunk is loaded with its first step; two chunks of two steps are in flight at once with four stages
    constexpr int NH = CK == 2 && ST == 4 ? 2 : 1;
    WHead<F> head[NH];
    auto wload = [&](auto uc, int it, WQ<F>& r) {      // uc: it % 4
        constexpr int U = decltype(uc)::value;
        const int t = kstep(it);
        const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc((void*)wbase, 0, t < nk ? (int)wbytes : 0, 0x00020000);
        if constexpr (U % CK == 0) wh_load<F, CK>(b, woff, h16, K, (uint32_t)t, head[(U >> 1) % NH]);
        wq_load<F>(b, woff, h16, (uint32_t)t, r);
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
    WDec<F, CK> dec;
    issue(std::integral_constant<int, 0>(), 0, 0, ND);
    __builtin_amdgcn_sched_barrier(0);
    wload(std::integral_constant<int, 0>(), 0, raw[0]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ST == 4) {
        issue(std::integral_constant<int, 1>(), 1, 0, ND);
        __builtin_amdgcn_sched_barrier(0);
        wload(std::integral_constant<int, 1>(), 1, raw[1]);
        __builtin_amdgcn_sched_barrier(0);
        issue(std::integral_constant<int, 2>(), 2, 0, ND);
        __builtin_amdgcn_sched_barrier(0);
        wload(std::integral_constant<int, 2>(), 2, raw[2]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Loads land in order, so a step's weight bytes in registers mean that the A stage issued before them has
    // landed too.  With four stages the stage after the current one is complete at each barrier, so its
    // first fragments are read a step early.
    constexpr bool kAhead = ST == 4;
    wq_landed<F>(raw[kAhead ? 1 : 0]);
    gt_barrier();
    wh_decode<F, CK>(head[0], kstep(0), nk, h, dec);
    gt_bf16x8 wv = w_slice<F, CK>(raw[0], dec, kstep(0), 0, 0), af[NRB], afn[NRB];
    if constexpr (kAhead) frags(std::integral_constant<int, 0>(), 0, af);
    // step `it` in stage S: four slices' MFMAs, each beside the dequantisation of the slice after it.  DMA and then
    // weight loads of step it + PF go out on the way (into the stage that step it - 1 read): with four stages one
    // part behind each slice, since all waves' loads at once stall on the address units; with two at once.
    auto body = [&](auto uc, int it) {                 // uc: it % 4
        constexpr int U = decltype(uc)::value, S = U % ST, P = (S + PF) % ST, Nx = (S + 1) % ST, UP = (U + PF) % 4, UN = (U + 1) % 4;
        const std::integral_constant<int, S> sc;
        if constexpr (!kAhead) {
            issue(std::integral_constant<int, P>(), it + PF, 0, ND);
            __builtin_amdgcn_sched_barrier(0);
            wload(std::integral_constant<int, UP>(), it + PF, raw[P]);
            __builtin_amdgcn_sched_barrier(0);
            frags(sc, 0, af);
        }
        const int t = kstep(it), t1 = kstep(it + 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) frags(sc, s + 1, afn);
            else if constexpr (kAhead) frags(std::integral_constant<int, Nx>(), 0, afn);
            gt_bf16x8 wn;
            if (s < 3) {
                wn = w_slice<F, CK>(raw[S], dec, t, U % CK, s + 1);
            } else {
                if constexpr (UN % CK == 0) wh_decode<F, CK>(head[(UN >> 1) % NH], t1, nk, h, dec);
                wn = w_slice<F, CK>(raw[Nx], dec, t1, UN % CK, 0);
            }
#pragma unroll
            for (int i = 0; i < NRB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], wv, acc[i], 0, 0, 0);
            constexpr int kV = (F == QMM_W_BF16 ? 0 : F == QMM_Q4_K ? 20 : 36) / NRB + 1;
#pragma unroll
            for (int i = 0; i < NRB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, kV, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kAhead) {
                if (s == 0) issue(std::integral_constant<int, P>(), it + PF, 0, (ND + 1) / 2);
                if (s == 1) issue(std::integral_constant<int, P>(), it + PF, (ND + 1) / 2, ND);
                if (s == 2) wload(std::integral_constant<int, UP>(), it + PF, raw[P]);
                __builtin_amdgcn_sched_barrier(0);
            }
            wv = wn;
#pragma unroll
            for (int i = 0; i < NRB; ++i) af[i] = afn[i];
        }
        wq_landed<F>(raw[kAhead ? (S + 2) % ST : Nx]);
        gt_barrier();
    };
    int it = 0;
    for (; it + 4 <= nit; it += 4) {
        body(std::integral_constant<int, 0>(), it);
        body(std::integral_constant<int, 1>(), it + 1);
        body(std::integral_constant<int, 2>(), it + 2);
        body(std::integral_constant<int, 3>(), it + 3);
    }
    if (it < nit) body(std::integral_constant<int, 0>(), it);
    if (it + 1 < nit) body(std::integral_constant<int, 1>(), it + 1);
    if (it + 2 < nit) body(std::integral_constant<int, 2>(), it + 2);
    __builtin_amdgcn_s_waitcnt(0);            // DMA of steps past the end
    if constexpr (std::is_invocable_v<const Put&, gt_f32x16 (&)[NRB]>) {      // the caller takes all registers at once
        put(acc);
    } else if constexpr (KS == 1) {
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
__device__ __forceinline__ void gemm_tile(const GemmArgs& a) {
    constexpr int BM = 32 * NRB, BN = 32 * CW;
    constexpr int kStage = KS * BM * 8;                        // 16-byte slots per stage, all K groups
    __shared__ uint4 s0[kStage], s1[kStage], s2[ST == 4 ? kStage : 1], s3[ST == 4 ? kStage : 1];
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    int tm, tn;
    gt_tile(blockIdx.x, mt * nt, mt, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int ncol = 32 * ((int)(threadIdx.x >> 6) % CW) + (lane & 31), n = n0 + ncol;
    // both operands through buffer resources over the tile's rows: rows past M or N are out of range and read
    // zeros without a memory access, and the DMA into LDS in this form leaves the compiler's count of
    // outstanding loads exact (the flat form makes it wait for all of them)
    const uint32_t abytes = (uint32_t)(min(BM, a.M - m0) - 1) * a.lda + 2u * (uint32_t)a.K;
    const uint32_t wbytes = (uint32_t)(min(BN, a.N - n0) - 1) * a.ldw + a.rowbytes;
    gemm_tile_core<F, NRB, CW, KS, ST>(
        s0, s1, s2, s3, a.A + (size_t)m0 * a.lda, abytes, a.W + (size_t)n0 * a.ldw, wbytes, a.ldw, a.K,
        [&](int r) { return (uint32_t)r * a.lda; },
        [&](int i, int e, float v) {
            const int m = m0 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
            if (m < a.M && n < a.N) {
                if constexpr (OUT_BF16) ((uint16_t*)a.D)[(size_t)m * a.ldd + n] = (uint16_t)f2bf_bits(v);
                else ((float*)a.D)[(size_t)m * a.ldd + n] = v;
            }
        });
}

template <int F, int NRB, int CW, int KS, int ST, bool OUT_BF16>
__global__ void __launch_bounds__(64 * CW * KS) k_gemm_tile(GemmArgs a) {
    gemm_tile<F, NRB, CW, KS, ST, OUT_BF16>(a);
}

}  // namespace qmm
