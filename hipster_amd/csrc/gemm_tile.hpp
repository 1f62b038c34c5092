// gemm_tile.hpp -- the prefill GEMM's kernels, D[m][n] = sum_k A[m][k] * bf16(W[n][k]), for every weight
// source of the call surface (Q4_K, Q5_K, IQ4_XS, Q6_K_SOA, Q8_0_SOA, Q5_1_SOA blocks and bf16 rows).
//
// Every output element is one chain of matrix instructions over K, k ascending, whatever the kernel, tile, weight source
// and shape: its bits depend on its own row and column only.  (Tiles whose waves took every eighth, fourth or second
// chunk of K and added their sums at the end were faster at few rows, 40 x 1024 x 5120 8.7 us against 9.2, 1 x 5120 x
// 17408 24 against 37, but gave other bits for other M and N.)
//
// k_gemm_tile: a workgroup computes a tile of 32 NRB rows x 32 CW columns with CW waves.  Wave cw owns the 32
// weight rows of its column block: it loads their quantised bytes straight into registers, dequantises them into the MFMA
// operand (every weight once per row tile, no LDS round trip) and multiplies them with all NRB row blocks of A, which the
// CW waves share through a ring of four LDS stages filled by DMA three steps ahead.  k_gemm_few, for few tiles, at the end.
//
// Which k a lane holds within a step is free as long as A and W agree: lane (r = l % 32, h = l / 32) of
// v_mfma_f32_32x32x16_bf16 supplies 8 values of its row per 16-wide slice, and the four slices of a
// step take them from 16-byte runs of quantised bytes that are contiguous in memory for that lane,
// so a step of 32 rows is one or two 16-byte loads per lane in every format.
//
// Measured against the 256 x 256 kernel it replaced, which dequantised through LDS and whose flat-form DMA made
// the compiler wait for every load in flight twice a step (calls in a stream, weights rotated, us):
//   M x N x K              Q4_K         Q6_K         Q8_0         bf16
//   2048 x 17408 x 5120    383 -> 327   681 -> 369   585 -> 347   503 -> 374
//   2048 x 5120 x 17408    485 -> 322   752 -> 387   659 -> 354   566 -> 390
//   300 x 17408 x 5120     135 -> 68    234 -> 89    201 -> 77    168 -> 97
//   300 x 5120 x 17408     415 -> 116   729 -> 122   641 -> 112   528 -> 108
//   40 x 1024 x 5120       119 -> 9     202 -> 14    162 -> 10    136 -> 9
// What bounds it (counters).  With many rows the card's power: 2048 x 17408 x 5120 Q4_K keeps the matrix cores busy 67% of the
// time at 1.57 GHz.  With few rows the vector memory path: the address units are busy 47% (300 x 17408 x 5120) to 76% (300 x
// 5120 x 17408 Q6_K, k_gemm_few) of the time at 34 cycles an instruction, since a load of one row per lane keeps them about as
// long whatever its width; without the weight loads the first took 53 us instead of 73 (no dequantisation 62, no
// matrix instructions 59, eight stages instead of four the same).  Hence the scales and high bits of four steps in one
// load (a step's loads Q4_K 2 -> 1.25, Q5_K 3 -> 1.5, Q6_K 4 -> 2, Q5_1 4 -> 2) and the loads of a step spread over its
// slices.  Measured and not kept: the weight rows through LDS by DMA with consecutive lanes on consecutive bytes (the same
// times: the LDS traffic and the waits took back what the address units gained), six and eight stages.
#pragma once
#include <type_traits>

#include "fmt_dequant.hpp"
#include "qmm_common.hpp"

namespace qmm {

constexpr int QMM_W_BF16 = 100;      // weight source: plain bf16 rows (not a wire format)

typedef __bf16 gt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gt_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 gt_h2 __attribute__((ext_vector_type(2)));

// A K step holds k = 64t .. 64t + 63, and lane half h supplies k = 32b + 16h .. + 15 of its sub-blocks b = 0, 1: slices
// 0, 1 take the first's two runs of 8, slices 2, 3 the second's.  A's 16-byte chunk (8 values of k) of slice s is
// therefore 4 (s / 2) + 2h + s % 2.  Every weight source gives its lanes these weights, so an output
// element is the same chain of matrix instructions whatever the format holding the weights.
__device__ __forceinline__ int a_chunk(int s, int h) { return 4 * (s >> 1) + 2 * h + (s & 1); }

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

// A lane's weights of one step: its quants (WQ), and the block's scales and high bits, loaded once per chunk of CK
// steps (WHead) and decoded for all of them at once (WDec): loads are what few rows cost, and a scale byte at a fixed
// place decodes in one instruction.
template <int F>
struct WQ {
    uint4 q;
    uint4 x;          // Q8_0, Q6_K: the second sub-block's
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
constexpr int CK = 4;         // steps of a chunk: a block of the 256-weight formats
// weights of step u of the chunk: fma(q, a[u], c[u]) in slices 0, 1 and fma(q, a2[u], c2[u]) in slices 2, 3 (q a
// whole number in an f16; where it is held as a subnormal, a carries the factor 2^24 or 2^20)
struct WDec {
    float a[CK], c[CK], a2[CK], c2[CK];
    uint4 hi[2];              // Q5_K: qh in hi[0]; Q6_K: qh of the halves
    uint32_t qh[CK];          // Q5_1: the lane's 16 bits of the first sub-block, then of the second
};

// w: the lane's row in the tile in bytes, h16 = 16 h, t the K step (uniform).  A Q6_K step is the low (t even) or high
// nibbles of two ql runs that its pair of steps shares: U = t % 4 says which is loaded, the first run at the even step, the
// second at the odd step before it (so that every step of the ring has a load behind its DMA).
template <int F, int U>
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
        if constexpr (U & 1) r.x = bld16(b, w + h16, 32u * t + 64u);
        else r.q = bld16(b, w + h16, 32u * t);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        r.q = bld16(b, w + h16, 64u * t);
        r.x = bld16(b, w + h16 + 32, 64u * t);
    } else {
        r.q = bld16(b, w + h16, 32u * t);
    }
}
// t0: the chunk's first step, a multiple of CK.  A partial chunk of d or m (K not in whole blocks of 256) reads up to 12 bytes
// past its row, for the matrix's last row past the matrix: the step is in the vector offset there, which the resource's
// range check counts by definition, dword by dword (gfx950 counts the scalar offset too).
template <int F>
__device__ __forceinline__ void wh_load(__amdgpu_buffer_rsrc_t b, uint32_t w, uint32_t h16, int K, uint32_t t0, WHead<F>& r) {
    const uint32_t nb = (uint32_t)K >> 8, k8 = (uint32_t)K >> 3, n = t0 >> 2;
    if constexpr (F == QMM_Q4_K) {
        r.x = bld16(b, w, n * 144u);
    } else if constexpr (F == QMM_Q5_K) {
        r.x = bld16(b, w, n * 176u);
        r.y[0] = bld16(b, w + h16, n * 176u + 16u);
    } else if constexpr (F == QMM_IQ4_XS) {
        r.sc = bld8(b, w, n * 136u);
    } else if constexpr (F == QMM_Q6_K_SOA) {
        r.x = bld16(b, w, nb * 192u + 16u * n);
        r.y[0] = bld16(b, w + h16, nb * 128u + 64u * n);
        r.y[1] = bld16(b, w + h16, nb * 128u + 64u * n + 32u);
        r.d = bld2(b, w, nb * 208u + 2u * n);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        r.x = bld16(b, w + (uint32_t)K + 4u * t0, 0);
    } else if constexpr (F == QMM_Q5_1_SOA) {
        r.x = bld16(b, w + 5u * k8 + 4u * t0, 0);
        r.m = bld16(b, w + 5u * k8 + (k8 >> 1) + 4u * t0, 0);
        r.y[0] = bld16(b, w, 4u * k8 + 8u * t0);
        r.y[1] = bld16(b, w, 4u * k8 + 8u * t0 + 16u);
    }
}

// byte i of word w as a float (i known at compile time: one instruction)
__device__ __forceinline__ float ub(uint32_t w, int i) { return (float)((w >> (8 * i)) & 0xffu); }
__device__ __forceinline__ uint32_t word(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// t0 as in wh_load.  Steps from nk on belong to no weight (their bytes are other data) and get scales of zero, by a mask:
// a select became control flow over whole steps.
template <int F>
__device__ __forceinline__ void wh_decode(const WHead<F>& r, int t0, int nk, int h, WDec& o) {
    if constexpr (F == QMM_Q4_K || F == QMM_Q5_K) {
        const float d = h2f(r.x.x), dmin = h2f(r.x.x >> 16);
        const float d24 = d * 16777216.f, dhi = d * (F == QMM_Q4_K ? 1048576.f : 16777216.f), nm = -dmin;
        const Q4kScaleBytes sb = q4k_scale_bytes(r.x.y, r.x.z, r.x.w);
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t s = u < 2 ? sb.sc_lo : sb.sc_hi, m = u < 2 ? sb.m_lo : sb.m_hi;
            o.a[u] = d24 * ub(s, 2 * (u & 1));
            o.c[u] = nm * ub(m, 2 * (u & 1));
            o.a2[u] = dhi * ub(s, 2 * (u & 1) + 1);
            o.c2[u] = nm * ub(m, 2 * (u & 1) + 1);
        }
        if constexpr (F == QMM_Q5_K) o.hi[0] = r.y[0];
    } else if constexpr (F == QMM_IQ4_XS) {
        const float d = h2f(r.sc.x);
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t sl = r.sc.y >> (8 * u), sh = r.sc.x >> (16 + 4 * u);
            o.a[u] = d * (float)((int)((sl & 15u) | ((sh & 3u) << 4)) - 32);
            o.a2[u] = d * (float)((int)(((sl >> 4) & 15u) | (((sh >> 2) & 3u) << 4)) - 32);
        }
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const float d = h2f(r.d);
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t s = word(r.x, u) >> (8 * h);
            o.a[u] = d * (float)(int8_t)s;
            o.a2[u] = d * (float)(int8_t)(s >> 16);
        }
        o.hi[0] = r.y[0];
        o.hi[1] = r.y[1];
    } else if constexpr (F == QMM_Q8_0_SOA) {
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t v = word(r.x, u) & (uint32_t)((t0 + u - nk) >> 31);
            o.a[u] = h2f(v);
            o.a2[u] = h2f(v >> 16);
        }
    } else if constexpr (F == QMM_Q5_1_SOA) {
#pragma unroll
        for (int u = 0; u < CK; ++u) {
            const uint32_t live = (uint32_t)((t0 + u - nk) >> 31), v = word(r.x, u) & live, m = word(r.m, u) & live;
            o.a[u] = h2f(v) * 16777216.f;
            o.a2[u] = h2f(v >> 16) * 16777216.f;
            o.c[u] = h2f(m);
            o.c2[u] = h2f(m >> 16);
            const uint4 y = r.y[u >> 1];
            const uint32_t y0 = u & 1 ? y.z : y.x, y1 = u & 1 ? y.w : y.y;
            o.qh[u] = __builtin_amdgcn_perm(y1, y0, h ? 0x07060302u : 0x05040100u);      // half h of each word
        }
    }
}

// The raw quants of a step as its slices read them: q the first sub-block's, x the second's.  IQ4_XS and Q5_1 pack
// weights l and l + 16 of a sub-block in a byte and lane half h loaded sub-block h: an exchange between the halves gives
// each its 16 weights of both sub-blocks (the first's high nibbles against the second's low ones), one per byte.
// In two parts, the words of slices 0, 2 and those of slices 1, 3.
template <int F, int PART>
__device__ __forceinline__ void wq_open(const WQ<F>& r, WQ<F>& o) {
    if constexpr (F == QMM_IQ4_XS || F == QMM_Q5_1_SOA) {
        auto swap = [](uint32_t v, uint32_t& a, uint32_t& b) {
            const auto s = __builtin_amdgcn_permlane32_swap(v & 0x0f0f0f0fu, (v >> 4) & 0x0f0f0f0fu, false, false);
            a = s[0];
            b = s[1];
        };
        if constexpr (PART == 0) {
            swap(r.q.x, o.q.x, o.x.x);
            swap(r.q.y, o.q.y, o.x.y);
        } else {
            swap(r.q.z, o.q.z, o.x.z);
            swap(r.q.w, o.q.w, o.x.w);
        }
    } else if constexpr (PART == 0) {
        o = r;
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
// four bytes b -> bf16(s * (b - bias)): b as the f16 number 1024 + b (one byte permute a pair), exactly, minus 1024 + bias
__device__ __forceinline__ void s4_bf16(uint32_t v, float s, float bias, gt_bf16x8& o, int i) {
    const gt_h2 k = {(_Float16)(1024.f + bias), (_Float16)(1024.f + bias)};
    const uint32_t e = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gt_h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)) - k);
    const uint32_t d = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gt_h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)) - k);
    o[i] = (__bf16)mix_lo(e, s, 0.f);
    o[i + 1] = (__bf16)mix_lo(d, s, 0.f);
    o[i + 2] = (__bf16)mix_hi(e, s, 0.f);
    o[i + 3] = (__bf16)mix_hi(d, s, 0.f);
}

// slice s of step u of the chunk: the lane's 8 weights, as qmm_dequant_bf16 gives them
template <int F>
__device__ __forceinline__ gt_bf16x8 w_slice(const WQ<F>& r, const WDec& c, int u, int s) {
    gt_bf16x8 o;
    if constexpr (F == QMM_W_BF16) {
        o = __builtin_bit_cast(gt_bf16x8, r.v[s]);
    } else if constexpr (F == QMM_Q4_K) {
        const uint32_t u0 = s & 1 ? r.q.z : r.q.x, u1 = s & 1 ? r.q.w : r.q.y;
        o = s < 2 ? q4_bf16x8_mix(u0, u1, 0x000f000fu, c.a[u], c.c[u]) : q4_bf16x8_mix(u0, u1, 0x00f000f0u, c.a2[u], c.c2[u]);
    } else {
        const float a = s < 2 ? c.a[u] : c.a2[u];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int w = 2 * (s & 1) + i;
            const uint32_t q = word(F != QMM_Q5_K && s >= 2 ? r.x : r.q, w);
            if constexpr (F == QMM_Q5_K) {
                const uint32_t nib = (s < 2 ? q : q >> 4) & 0x0f0f0f0fu;
                const uint32_t v = nib | (((word(c.hi[0], w) >> (2 * u + (s >> 1))) & 0x01010101u) << 4);
                u4_bf16(v, a, s < 2 ? c.c[u] : c.c2[u], o, 4 * i);
            } else if constexpr (F == QMM_IQ4_XS) {
                s4_bf16(iq4_levels4(q, 0x80808080u), a, 128.f, o, 4 * i);
            } else if constexpr (F == QMM_Q6_K_SOA) {
                const uint32_t nib = (q >> (4 * (u & 1))) & 0x0f0f0f0fu;
                const uint32_t v = nib | (((word(c.hi[u >> 1], w) >> (4 * (u & 1) + 2 * (s >> 1))) & 0x03030303u) << 4);
                s4_bf16(v, a, 32.f, o, 4 * i);
            } else if constexpr (F == QMM_Q8_0_SOA) {
                s4_bf16(q ^ 0x80808080u, a, 128.f, o, 4 * i);
            } else {                                     // QMM_Q5_1_SOA: bits 16 (s / 2) + 4w .. + 3 of qh, one per byte
                const uint32_t hb = ((((c.qh[u] >> (16 * (s >> 1) + 4 * w)) & 0xfu) * 0x00204081u) & 0x01010101u) << 4;
                u4_bf16(q | hb, a, s < 2 ? c.c[u] : c.c2[u], o, 4 * i);
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

struct GemmArgs {
    const uint8_t* A;          // bf16 rows, lda bytes apart
    const uint8_t* W;          // weight rows, ldw bytes apart
    void* D;                   // f32 or bf16, rows ldd elements apart
    uint32_t lda, ldw, rowbytes;   // rowbytes: a weight row's own bytes
    int M, N, K, ldd;
    uint32_t apast, wpast;     // byte offsets in a tile for its rows past M and N (launch_gemm)
};

// workgroup id -> tile: workgroup i runs on XCD i % 8, which takes a contiguous range of the tiles (M
// tiles fastest), so the M tiles that share weight rows share one L2
__device__ __forceinline__ void gt_tile(int bid, int ntiles, int mt, int& tm, int& tn) {
    const int x = bid & 7, q = ntiles >> 3, rem = ntiles & 7;
    const int id = x * q + (x < rem ? x : rem) + (bid >> 3);
    tm = id % mt;
    tn = id / mt;
}

template <int V>
using gt_ic = std::integral_constant<int, V>;

// Both operands go through buffer resources over the tile's rows: rows past M or N are out of range and read zeros
// without a memory access, and the DMA into LDS in this form leaves the compiler's count of outstanding loads exact
// (the flat form makes it wait for all of them).  K steps past the end read through an empty resource.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gt_rsrc(const uint8_t* base, uint32_t bytes, bool live) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, live ? (int)bytes : 0, 0x00020000);
}
__device__ __forceinline__ void gt_dma(__amdgpu_buffer_rsrc_t r, uint4* lds, uint32_t v, uint32_t s) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, v, s, 0, 0);
}

static __device__ const uint8_t gt_zeros[16] __attribute__((aligned(16))) = {};      // steps past the end for 64-bit row offsets

// One tile of 32 NRB rows x 32 CW columns, CW waves.  s0..s3: the ring's stages, at least 32 NRB * 8 slots each and separate __shared__ arrays: the compiler then knows which stage a DMA writes and an LDS read
// waits for that stage only.  abase / wbase: the operands' tile, abytes / wbytes its extent; arow(r), woff: byte offsets of
// A's row r and of the lane's weight row (column 32 cw + fr) in it (64-bit offsets of A go past the resource); put(i, e, v): register e of row block i, which is row 32i + 8(e/4) + 4h + e%4, column 32 cw + fr.
template <int F, int NRB, int CW, class ARow, class Put>
__device__ __forceinline__ void gemm_tile_core(uint4* s0, uint4* s1, uint4* s2, uint4* s3, const uint8_t* abase, uint32_t abytes,
                                               const uint8_t* wbase, uint32_t wbytes, uint32_t woff, int K, const ARow& arow,
                                               const Put& put) {
    constexpr int NI = 4 * NRB, ND = (NI + CW - 1) / CW;
    const int lane = threadIdx.x & 63, fr = lane & 31, h = lane >> 5, fx = (fr >> 1) & 7;
    const int cw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nk = K >> 6;
    const uint32_t h16 = 16u * (uint32_t)h;
    // DMA instruction q of the stage fills slots 64q + lane: rows 8q..8q+7, slot column lane % 8
    using Off = decltype(arow(0));       // uint64_t: rows beyond a buffer offset's span
    Off aoff[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int q = min(cw + CW * i, NI - 1), r = 8 * q + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        aoff[i] = arow(r) + 16u * (uint32_t)c;
    }
    auto stage = [&](auto sc) -> uint4* {
        constexpr int S = decltype(sc)::value;
        if constexpr (S == 0) return s0;
        else if constexpr (S == 1) return s1;
        else if constexpr (S == 2) return s2;
        else return s3;
    };
    auto issue = [&](auto sc, int t, int i0, int i1) {
        const __amdgpu_buffer_rsrc_t r = gt_rsrc(abase, abytes, t < nk);
        uint4* st = stage(sc);
#pragma unroll
        for (int i = 0; i < ND; ++i)
            if (i >= i0 && i < i1 && (NI % CW == 0 || cw + CW * i < NI)) {
                uint4* dst = st + 64 * (cw + CW * i);
                if constexpr (sizeof(Off) == 4) gt_dma(r, dst, aoff[i], 128u * (uint32_t)t);
                else dma16((t < nk ? abase + 128u * (uint32_t)t : gt_zeros) + (t < nk ? aoff[i] : 0), lds_addr(dst));
            }
    };
    WQ<F> raw[4];
    WHead<F> head;                                     // loaded with the first step of its chunk
    auto wload = [&](auto uc, int t, WQ<F>& r) {       // uc: t % 4
        constexpr int U = decltype(uc)::value;
        const __amdgpu_buffer_rsrc_t b = gt_rsrc(wbase, wbytes, t < nk);
        if constexpr (U == 0) wh_load<F>(b, woff, h16, K, (uint32_t)t, head);
        wq_load<F, U>(b, woff, h16, (uint32_t)t, r);
    };
    // a use of a step's weights: its loads, and the DMA issued before them, have landed here
    auto landed = [&](auto uc) {                       // uc: t % 4
        constexpr int U = decltype(uc)::value;
        const WQ<F>& r = raw[U];
        if constexpr (F == QMM_W_BF16) asm volatile("" ::"v"(r.v[0].x), "v"(r.v[1].x), "v"(r.v[2].x), "v"(r.v[3].x));
        else if constexpr (F == QMM_Q8_0_SOA) asm volatile("" ::"v"(r.q.x), "v"(r.x.x));
        else if constexpr (F == QMM_Q6_K_SOA && (U & 1)) asm volatile("" ::"v"(r.x.x));
        else asm volatile("" ::"v"(r.q.x));
    };
    WQ<F> cur;                                         // the current step's weights
    auto open = [&](auto uc) {                         // uc: t % 4
        constexpr int U = decltype(uc)::value;
        if constexpr (F == QMM_Q6_K_SOA) {             // a pair of steps: its second run came with the step before
            if constexpr ((U & 1) == 0) {
                cur.q = raw[U].q;
                cur.x = raw[(U + 3) % 4].x;
            }
        } else {
            wq_open<F, 0>(raw[U], cur);
        }
    };
    auto frags = [&](auto sc, int s, gt_bf16x8 (&af)[NRB]) {
        const uint4* la = stage(sc);
#pragma unroll
        for (int i = 0; i < NRB; ++i) {
            const uint4 v = la[(32 * i + fr) * 8 + (a_chunk(s, h) ^ fx)];
            af[i] = __builtin_bit_cast(gt_bf16x8, v);
        }
    };
    gt_f32x16 acc[NRB];
#pragma unroll
    for (int i = 0; i < NRB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
    // prologue: steps 0, 1, 2 in flight
    WDec dec;
    if constexpr (F == QMM_Q6_K_SOA) raw[3].x = bld16(gt_rsrc(wbase, wbytes, true), woff + h16, 32u);
    auto first = [&](auto uc) {
        constexpr int U = decltype(uc)::value;
        issue(uc, U, 0, ND);
        __builtin_amdgcn_sched_barrier(0);
        wload(uc, U, raw[U]);
        __builtin_amdgcn_sched_barrier(0);
    };
    first(gt_ic<0>());
    first(gt_ic<1>());
    first(gt_ic<2>());
    // Loads land in order, so a step's weight bytes in registers mean that the A stage issued before them has landed too.
    // The stage after the current one is complete at each barrier, so its first fragments are read a step early.
    landed(gt_ic<1>());
    gt_barrier();
    wh_decode<F>(head, 0, nk, h, dec);
    open(gt_ic<0>());
    gt_bf16x8 wv = w_slice<F>(cur, dec, 0, 0), af[NRB], afn[NRB];
    frags(gt_ic<0>(), 0, af);
    // step t in stage S = t % 4: four slices' MFMAs, each beside the dequantisation of the slice after it.  DMA and then weight
    // loads of step t + 3 go out on the way (into the stage that step t - 1 read), one part behind each slice, since all
    // waves' loads at once stall on the address units.
    auto body = [&](auto uc, int t) {                  // uc: t % 4
        constexpr int U = decltype(uc)::value, P = (U + 3) % 4, UN = (U + 1) % 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) frags(uc, s + 1, afn);
            else frags(gt_ic<UN>(), 0, afn);
            gt_bf16x8 wn;
            if (s < 3) {
                if (s == 0) wq_open<F, 1>(raw[U], cur);
                wn = w_slice<F>(cur, dec, U, s + 1);
            } else {
                if constexpr (UN == 0) wh_decode<F>(head, t + 1, nk, h, dec);
                open(gt_ic<UN>());
                wn = w_slice<F>(cur, dec, UN, 0);
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
            if (s == 0) issue(gt_ic<P>(), t + 3, 0, (ND + 1) / 2);
            if (s == 1) issue(gt_ic<P>(), t + 3, (ND + 1) / 2, ND);
            if (s == 2) wload(gt_ic<P>(), t + 3, raw[P]);
            __builtin_amdgcn_sched_barrier(0);
            wv = wn;
#pragma unroll
            for (int i = 0; i < NRB; ++i) af[i] = afn[i];
        }
        landed(gt_ic<(U + 2) % 4>());
        gt_barrier();
    };
    // In fours: steps past the last (K not in whole blocks of 256) add zeros from empty resources, with scales of zero.  A
    // tail of its own, or a way out of the loop, made the compiler keep a second set of registers (up to 800
    // spilled) or wait for every load in flight once a round.
    for (int t = 0; t < nk; t += 4) {
        body(gt_ic<0>(), t);
        body(gt_ic<1>(), t + 1);
        body(gt_ic<2>(), t + 2);
        body(gt_ic<3>(), t + 3);
    }
    __builtin_amdgcn_s_waitcnt(0);            // DMA of steps past the end
    if constexpr (std::is_invocable_v<const Put&, gt_f32x16 (&)[NRB]>) {      // the caller takes all registers at once
        put(acc);
    } else {
#pragma unroll
        for (int i = 0; i < NRB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) put(i, e, acc[i][e]);
    }
}

template <bool OUT_BF16>
__device__ __forceinline__ void gt_put(const GemmArgs& a, int m, int n, float v) {
    if (m < a.M && n < a.N) {
        if constexpr (OUT_BF16) ((uint16_t*)a.D)[(size_t)m * a.ldd + n] = (uint16_t)f2bf_bits(v);
        else ((float*)a.D)[(size_t)m * a.ldd + n] = v;
    }
}

template <int F, int NRB, int CW, bool OUT_BF16>
__global__ void __launch_bounds__(64 * CW) k_gemm_tile(GemmArgs a) {
    constexpr int BM = 32 * NRB, BN = 32 * CW, kStage = BM * 8;           // 16-byte slots per stage
    __shared__ uint4 s0[kStage], s1[kStage], s2[kStage], s3[kStage];
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    int tm, tn;
    gt_tile(blockIdx.x, mt * nt, mt, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN, lane = threadIdx.x & 63, h = lane >> 5, col = 32 * (int)(threadIdx.x >> 6) + (lane & 31);
    const int rows = min(BM, a.M - m0), cols = min(BN, a.N - n0);
    gemm_tile_core<F, NRB, CW>(
        s0, s1, s2, s3, a.A + (size_t)m0 * a.lda, (uint32_t)(rows - 1) * a.lda + 2u * (uint32_t)a.K, a.W + (size_t)n0 * a.ldw,
        (uint32_t)(cols - 1) * a.ldw + a.rowbytes, col < cols ? (uint32_t)col * a.ldw : a.wpast, a.K,
        [&](int r) { return r < rows ? (uint32_t)r * a.lda : a.apast; },
        [&](int i, int e, float v) { gt_put<OUT_BF16>(a, m0 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3), n0 + col, v); });
}

// ------------------------------------------------------------------------------------------
// Few tiles (M x N small): there a wave per 32 columns dequantises and multiplies in turn, and its chain over K has no other
// wave to hide behind.  Here P producer waves dequantise the 64-wide steps of a batch side by side into LDS, bring
// A by DMA, and consumer waves run the chains of matrix instructions over both, in the order of k.
// v_mfma_f32_16x16x32_bf16 adds its four runs of 8 in two halves as two v_mfma_f32_32x32x16_bf16 do, so a lane group g
// = lane / 16 that supplies run 2 (g % 2) + g / 2 of a sub-block gives the tile kernel's bits.  A producer's unit is 16
// weight rows of one step: half the dequantisation of a 32-row unit between two barriers, and tiles of 16 columns
// for matrices of few rows.

// A lane's weights of a unit: 8 of each sub-block of the step, k = 32b + 8c .. + 7 (c = the run above).  A load costs the
// address units about the same whatever its width, so each is as wide as a row's four lanes can share, and what a lane
// does not hold itself comes by swaps between the lane groups (u_open).
template <int F>
struct UQ {
    uint2 q[2];           // opened: per sub-block (Q4_K, Q5_K: q[0] holds both; Q6_K: shared by a pair of steps)
};
template <>
struct UQ<QMM_W_BF16> {
    uint4 v[2];
};
struct UHead {
    uint4 x;              // Q4_K, Q5_K: block header; Q6_K: scales of the pair's steps and d; Q8_0: d; Q5_1: d, m, qh (opened)
    uint2 h;              // Q5_K, Q6_K: high bits of the run; IQ4_XS: block header
};
// US steps from t (t even when US = 2: Q6_K, whose pair shares its loads); g = lane / 16
template <int F>
__device__ __forceinline__ void u_load(__amdgpu_buffer_rsrc_t b, uint32_t w, uint32_t g, uint32_t c, int K, uint32_t t, UQ<F>& r, UHead& hd) {
    const uint32_t nb = (uint32_t)K >> 8, k8 = (uint32_t)K >> 3, j = t & 3, n = t >> 2;
    if constexpr (F == QMM_W_BF16) {
        r.v[0] = bld16(b, w + 16 * c, 128u * t);
        r.v[1] = bld16(b, w + 16 * c + 64, 128u * t);
    } else if constexpr (F == QMM_Q4_K) {
        hd.x = bld16(b, w, n * 144u);
        r.q[0] = bld8(b, w + 8 * c, n * 144u + 16u + 32u * j);
    } else if constexpr (F == QMM_Q5_K) {
        hd.x = bld16(b, w, n * 176u);
        hd.h = bld8(b, w + 8 * c, n * 176u + 16u);
        r.q[0] = bld8(b, w + 8 * c, n * 176u + 48u + 32u * j);
    } else if constexpr (F == QMM_IQ4_XS) {
        hd.h = bld8(b, w, n * 136u);
        r.q[0] = bld8(b, w + 16 * (g & 1) + 8 * (g >> 1), n * 136u + 8u + 32u * j);
    } else if constexpr (F == QMM_Q6_K_SOA) {
        // groups 0, 1: the scales of steps t, t + 1; groups 2, 3: the dword with d
        hd.x.x = bld4(b, w + (g < 2 ? nb * 192u + 4u * (t + g) : nb * 208u + ((2u * n) & ~3u)), 0);
        hd.h = bld8(b, w + 8 * c, nb * 128u + 16u * t);
        r.q[0] = bld8(b, w + 8 * c, 32u * t);
        r.q[1] = bld8(b, w + 8 * c + 32, 32u * t);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        hd.x.x = bld4(b, w, (uint32_t)K + 4u * t);
        const uint4 v = bld16(b, w + 32 * (g >> 1) + 16 * (g & 1), 64u * t);
        r.q[0] = make_uint2(v.x, v.y);
        r.q[1] = make_uint2(v.z, v.w);
    } else {
        // groups 0 .. 3: d, m, and the two words of qh
        hd.x.x = bld4(b, w + (g == 0 ? 5u * k8 : g == 1 ? 5u * k8 + (k8 >> 1) : 4u * k8 + 4u * (g - 2)) + (g < 2 ? 4u : 8u) * t, 0);
        r.q[0] = bld8(b, w + 16 * (g & 1) + 8 * (g >> 1), 32u * t);
    }
}
// v of groups 0 and 2 in a, of groups 1 and 3 in b, for the pairs of groups (0, 1) and (2, 3)
__device__ __forceinline__ void u_pairs(uint32_t v, uint32_t& a, uint32_t& b) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    a = s[0];
    b = s[1];
}
__device__ __forceinline__ void u_halves(uint32_t v, uint32_t& a, uint32_t& b) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = s[0];
    b = s[1];
}
template <int F>
__device__ __forceinline__ void u_open(UQ<F>& r, UHead& hd) {
    if constexpr (F == QMM_IQ4_XS || F == QMM_Q5_1_SOA) {      // even groups loaded the first sub-block's bytes, odd ones the second's
        const uint2 v = r.q[0];
        u_pairs(v.x, r.q[0].x, r.q[1].x);
        u_pairs(v.y, r.q[0].y, r.q[1].y);
    }
    if constexpr (F == QMM_Q8_0_SOA) {      // groups 0, 1 loaded runs 0, 1 and 2, 3 of the first sub-block, groups 2, 3 of the second
        const auto s = __builtin_amdgcn_permlane32_swap(r.q[0].x, r.q[1].x, false, false);
        const auto t = __builtin_amdgcn_permlane32_swap(r.q[0].y, r.q[1].y, false, false);
        r.q[0] = make_uint2(s[0], t[0]);
        r.q[1] = make_uint2(s[1], t[1]);
    }
    if constexpr (F == QMM_Q6_K_SOA || F == QMM_Q5_1_SOA) {
        uint32_t e, o;
        u_pairs(hd.x.x, e, o);
        u_halves(e, hd.x.x, hd.x.z);
        u_halves(o, hd.x.y, hd.x.w);
    }
}
// step t (step u of the unit), sub-block b.  live: all ones, or zero for steps past the row's last
template <int F>
__device__ __forceinline__ gt_bf16x8 u_frag(const UQ<F>& r, const UHead& hd, uint32_t c, int t, int u, int b, uint32_t live) {
    gt_bf16x8 o;
    const int j = t & 3;
    if constexpr (F == QMM_W_BF16) {
        o = __builtin_bit_cast(gt_bf16x8, r.v[b]);
    } else if constexpr (F == QMM_Q4_K || F == QMM_Q5_K) {
        const Q4kScaleBytes sb = q4k_scale_bytes(hd.x.y, hd.x.z, hd.x.w);
        const int i = 16 * (j & 1) + 8 * b;
        const float sc = h2f(hd.x.x) * (float)(((j < 2 ? sb.sc_lo : sb.sc_hi) >> i) & 0xffu);
        const float m = -h2f(hd.x.x >> 16) * (float)(((j < 2 ? sb.m_lo : sb.m_hi) >> i) & 0xffu);
        if constexpr (F == QMM_Q4_K) {
            o = b == 0 ? q4_bf16x8_mix(r.q[0].x, r.q[0].y, 0x000f000fu, sc * 16777216.f, m)
                       : q4_bf16x8_mix(r.q[0].x, r.q[0].y, 0x00f000f0u, sc * 1048576.f, m);
        } else {
            const int hb = 2 * j + b;
            u4_bf16(((r.q[0].x >> (4 * b)) & 0x0f0f0f0fu) | (((hd.h.x >> hb) & 0x01010101u) << 4), sc * 16777216.f, m, o, 0);
            u4_bf16(((r.q[0].y >> (4 * b)) & 0x0f0f0f0fu) | (((hd.h.y >> hb) & 0x01010101u) << 4), sc * 16777216.f, m, o, 4);
        }
    } else if constexpr (F == QMM_IQ4_XS) {
        const uint32_t sl = hd.h.y >> (8 * j + 4 * b), sh = hd.h.x >> (16 + 4 * j + 2 * b), n = 4 * (c >> 1);
        const float sc = h2f(hd.h.x) * (float)((int)((sl & 15u) | ((sh & 3u) << 4)) - 32);
        s4_bf16(iq4_levels4((r.q[b].x >> n) & 0x0f0f0f0fu, 0x80808080u), sc, 128.f, o, 0);
        s4_bf16(iq4_levels4((r.q[b].y >> n) & 0x0f0f0f0fu, 0x80808080u), sc, 128.f, o, 4);
    } else if constexpr (F == QMM_Q6_K_SOA) {
        const float sc = h2f(hd.x.z >> (16 * ((t >> 2) & 1))) * (float)(int8_t)((u ? hd.x.y : hd.x.x) >> (16 * b + 8 * (c >> 1)));
        const int n = 4 * u, hb = 4 * u + 2 * b;
        s4_bf16(((r.q[b].x >> n) & 0x0f0f0f0fu) | (((hd.h.x >> hb) & 0x03030303u) << 4), sc, 32.f, o, 0);
        s4_bf16(((r.q[b].y >> n) & 0x0f0f0f0fu) | (((hd.h.y >> hb) & 0x03030303u) << 4), sc, 32.f, o, 4);
    } else if constexpr (F == QMM_Q8_0_SOA) {
        const float sc = h2f((hd.x.x & live) >> (16 * b));
        s4_bf16(r.q[b].x ^ 0x80808080u, sc, 128.f, o, 0);
        s4_bf16(r.q[b].y ^ 0x80808080u, sc, 128.f, o, 4);
    } else {
        const float sc = h2f((hd.x.x & live) >> (16 * b)) * 16777216.f, m = h2f((hd.x.y & live) >> (16 * b));
        const uint32_t n = 4 * (c >> 1), qh = (b ? hd.x.w : hd.x.z) >> (8 * c);
        auto hi = [](uint32_t v) { return (((v & 0xfu) * 0x00204081u) & 0x01010101u) << 4; };
        u4_bf16(((r.q[b].x >> n) & 0x0f0f0f0fu) | hi(qh), sc, m, o, 0);
        u4_bf16(((r.q[b].y >> n) & 0x0f0f0f0fu) | hi(qh >> 4), sc, m, o, 4);
    }
    return o;
}

typedef float gt_f32x4 __attribute__((ext_vector_type(4)));
template <int F>
constexpr int gf_us = F == QMM_Q6_K_SOA ? 2 : 1;
// R row blocks and CB column blocks of 16; a consumer takes CR x CC of them; B steps a batch
template <int F, int R, int CB, int CR, int CC, int B>
constexpr int gf_waves = B * CB / gf_us<F> + (R / CR) * (CB / CC);

template <int F, int R, int CB, int CR, int CC, int B, bool OUT_BF16>
__global__ void __launch_bounds__((64 * gf_waves<F, R, CB, CR, CC, B>)) k_gemm_few(GemmArgs a) {
    constexpr int BM = 16 * R, BN = 16 * CB, US = gf_us<F>, P = B * CB / US;
    static_assert(R % CR == 0 && CB % CC == 0 && B % US == 0, "");
    constexpr int kA = B * BM * 8, kW = B * CB * 128;          // slots per stage
    __shared__ uint4 As[4 * kA], Ws[2 * kW];
    const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
    int tm, tn;
    gt_tile(blockIdx.x, mt * nt, mt, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN, lane = threadIdx.x & 63, fr = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nk = a.K >> 6, nb = (nk + B - 1) / B;
    const uint32_t c = 2u * (g & 1) + (uint32_t)(g >> 1);
    if (wave < P) {
        const uint8_t* abase = a.A + (size_t)m0 * a.lda;
        const uint8_t* wbase = a.W + (size_t)n0 * a.ldw;
        const int rows = min(BM, a.M - m0), cols = min(BN, a.N - n0);
        const uint32_t abytes = (uint32_t)(rows - 1) * a.lda + 2u * (uint32_t)a.K, wbytes = (uint32_t)(cols - 1) * a.ldw + a.rowbytes;
        const int cb = wave % CB, st = (wave / CB) * US;       // this wave's column block and first step of a batch
        const uint32_t woff = 16 * cb + fr < cols ? (uint32_t)(16 * cb + fr) * a.ldw : a.wpast;
        constexpr int ND = 2 * R / CB;                         // A: 8-row runs cb, cb + CB, .. of the wave's own steps
        static_assert(2 * R % CB == 0, "");
        uint32_t aoff[ND];
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int r = 8 * (cb + CB * i) + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
            aoff[i] = (r < rows ? (uint32_t)r * a.lda : a.apast) + 16u * (uint32_t)ch;
        }
        UQ<F> raw[4];
        UHead head[4];
        auto wissue = [&](auto sc, int b) {                    // weights of batch b into registers b % 4
            constexpr int S = decltype(sc)::value;
            const int t = b * B + st;
            u_load<F>(gt_rsrc(wbase, wbytes, t < nk), woff, (uint32_t)g, c, a.K, (uint32_t)t, raw[S], head[S]);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto aissue = [&](auto sc, int b) {                    // A of batch b into stage b % 4
            constexpr int S = decltype(sc)::value;
#pragma unroll
            for (int u = 0; u < US; ++u) {
                const int t = b * B + st + u;
                const __amdgpu_buffer_rsrc_t r = gt_rsrc(abase, abytes, t < nk);
#pragma unroll
                for (int i = 0; i < ND; ++i) gt_dma(r, As + S * kA + (st + u) * BM * 8 + 64 * (cb + CB * i), aoff[i], 128u * (uint32_t)t);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto produce = [&](auto sc, int b) {
            constexpr int S = decltype(sc)::value;
            uint4* ws = Ws + (S & 1) * kW + (st * CB + cb) * 128 + lane;
            UQ<F> q = raw[S];
            UHead hd = head[S];
            u_open<F>(q, hd);
#pragma unroll
            for (int u = 0; u < US; ++u) {
                const int t = b * B + st + u;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    ws[u * CB * 128 + 64 * h] = __builtin_bit_cast(uint4, u_frag<F>(q, hd, c, t, u, h, (uint32_t)((t - nk) >> 31)));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // Loads land in order: the weights of batch b + 3 in registers mean that A's batch b + 1, issued before them, has landed
        // (all of them before the dequantisation: it waited for the address units, 49 -> 56 us at 40 x 5120 x 17408; all behind it: 52).
        auto landed = [&](auto sc) {
            const UQ<F>& r = raw[decltype(sc)::value];
            if constexpr (F == QMM_W_BF16) asm volatile("" ::"v"(r.v[0].x), "v"(r.v[1].x));
            else if constexpr (F == QMM_Q6_K_SOA || F == QMM_Q8_0_SOA) asm volatile("" ::"v"(r.q[0].x), "v"(r.q[1].x));
            else asm volatile("" ::"v"(r.q[0].x));
        };
        wissue(gt_ic<0>(), 0);
        aissue(gt_ic<0>(), 0);
        wissue(gt_ic<1>(), 1);
        aissue(gt_ic<1>(), 1);
        wissue(gt_ic<2>(), 2);
        aissue(gt_ic<2>(), 2);
        wissue(gt_ic<3>(), 3);
        produce(gt_ic<0>(), 0);
        landed(gt_ic<1>());                                    // A's batch 0
        gt_barrier();
        auto body = [&](auto sc, int b) {
            constexpr int S = decltype(sc)::value;
            wissue(gt_ic<S>(), b + 4);
            produce(gt_ic<(S + 1) % 4>(), b + 1);
            aissue(gt_ic<(S + 3) % 4>(), b + 3);               // the stage that batch b - 1 read
            landed(gt_ic<(S + 3) % 4>());
            gt_barrier();
        };
        for (int b = 0;; b += 4) {
            body(gt_ic<0>(), b);
            if (b + 1 == nb) break;
            body(gt_ic<1>(), b + 1);
            if (b + 2 == nb) break;
            body(gt_ic<2>(), b + 2);
            if (b + 3 == nb) break;
            body(gt_ic<3>(), b + 3);
            if (b + 4 == nb) break;
        }
        __builtin_amdgcn_s_waitcnt(0);        // DMA of steps past the end
    } else {                                                   // consumers
        const int con = wave - P, cb = (con % (CB / CC)) * CC, rb = (con / (CB / CC)) * CR;
        gt_f32x4 acc[CR][CC];
#pragma unroll
        for (int i = 0; i < CR; ++i)
#pragma unroll
            for (int k = 0; k < CC; ++k) acc[i][k] = gt_f32x4{0.f, 0.f, 0.f, 0.f};
        const uint4* la = As + (16 * rb + fr) * 8;
        const uint4* lw = Ws + cb * 128 + lane;
        const int fx = (fr >> 1) & 7;
        gt_barrier();
        for (int b = 0; b < nb; ++b) {
            const uint4* sa = la + (b & 3) * kA;
            const uint4* sw = lw + (b & 1) * kW;
            uint4 wf[2][CC], af[2][CR];
            auto read = [&](int x) {                           // sub-block x % 2 of step x / 2
#pragma unroll
                for (int k = 0; k < CC; ++k) wf[x & 1][k] = sw[(x >> 1) * CB * 128 + k * 128 + 64 * (x & 1)];
#pragma unroll
                for (int i = 0; i < CR; ++i) af[x & 1][i] = sa[(x >> 1) * BM * 8 + 128 * i + ((4 * (x & 1) + (int)c) ^ fx)];
            };
            read(0);
#pragma unroll
            for (int x = 0; x < 2 * B; ++x) {
                if (x + 1 < 2 * B) read(x + 1);
#pragma unroll
                for (int i = 0; i < CR; ++i)
#pragma unroll
                    for (int k = 0; k < CC; ++k)
                        acc[i][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gt_bf16x8, af[x & 1][i]),
                                                                            __builtin_bit_cast(gt_bf16x8, wf[x & 1][k]), acc[i][k], 0, 0, 0);
            }
            gt_barrier();
        }
#pragma unroll
        for (int i = 0; i < CR; ++i)
#pragma unroll
            for (int k = 0; k < CC; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) gt_put<OUT_BF16>(a, m0 + 16 * (rb + i) + 4 * g + e, n0 + 16 * (cb + k) + fr, acc[i][k][e]);
    }
}

}  // namespace qmm
