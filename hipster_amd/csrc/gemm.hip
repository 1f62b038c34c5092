// gemm.hip -- prefill-sized matrix products on gfx950: dequantisation to bf16, a Q4_K-weight GEMM
// with the dequantisation fused into the LDS staging of the weight tile, a plain bf16 GEMM and the
// bf16 <-> f32 helpers of the reference's engine/kernels/gemm.h.
//
// Entry points (C ABI, include/hipster_qmm.h) and the reference functions they replace:
//   qmm_dequant_bf16        hip::dequant_bf16     engine/kernels/gemm.hip:16-76,96-107
//   qmm_gemm_wq             (new) dequant_bf16 + BlasLt::gemm fused; engine/src/qwen35.cpp:204-239,
//                           engine/src/qwen4exp.cpp:513-527 are the callers it serves
//   qmm_gemm_bf16           hip::BlasLt::gemm     engine/kernels/gemm.hip:125-160 (own MFMA kernel, no hipBLASLt)
//   qmm_f32_to_bf16, qmm_bf16_to_f32, qmm_bf16_to_f32_seg, qmm_bf16_to_f32_seg2   gemm.hip:77-95
//
// qmm_gemm_wq and qmm_gemm_bf16 run the kernels of gemm_tile.hpp with the weight source as a template
// argument; pick_tile below chooses the tile by the shape.
#include "fmt_dequant.hpp"
#include "gemm_tile.hpp"
#include "qmm_common.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

namespace qmm {
namespace {

// ------------------------------------------------------------------------------------------
// Bit-exact dequantisation to bf16 (engine/src/quant.h:43-53,65-80 arithmetic, then RNE to bf16 as
// engine/kernels/gemm.hip:12).  Contraction is off: (d*sc)*q and dmin*m are rounded on their own,
// exactly as the host reference computes them.
#pragma clang fp contract(off)

// Q4_K: one thread per 32-weight sub-block (8 per block); writes 32 bf16 (64 B)
__global__ void __launch_bounds__(256) k_dequant_q4k_bf16(const uint8_t* __restrict__ W, uint16_t* __restrict__ out,
                                                          size_t nsub, int K) {
    const size_t g = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= nsub) return;
    const size_t blk = g >> 3;
    const int s = (int)(g & 7), j = s >> 1, h = s & 1;
    const uint8_t* bp = W + blk * 144;
    const uint4 hd = ld16(bp);
    const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
    const Q4kScaleBytes sb = q4k_scale_bytes(hd.y, hd.z, hd.w);
    const float dl = d * (float)byte8(sb.sc_lo, sb.sc_hi, s), ml = dmin * (float)byte8(sb.m_lo, sb.m_hi, s);
    const uint4 q0 = ld16(bp + 16 + 32 * j), q1 = ld16(bp + 32 + 32 * j);
    const uint32_t qw[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    uint32_t o[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t v = h ? (qw[i] >> 4) : qw[i];
        uint32_t bf[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) bf[b] = f2bf_bits(dl * (float)((v >> (8 * b)) & 15u) - ml);
        o[2 * i] = bf[0] | (bf[1] << 16);
        o[2 * i + 1] = bf[2] | (bf[3] << 16);
    }
    // element index of this sub-block: row-major [N][K] with K = nb * 256 -> block blk holds elements blk*256..
    uint4* dst = (uint4*)(out + blk * 256 + 32 * s);
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = make_uint4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
}

// Q6_K (GGUF 210-byte blocks, or the row-SoA repack): one thread per 16 weights sharing one scale
template <int F>
__global__ void __launch_bounds__(256) k_dequant_q6k_bf16(const uint8_t* __restrict__ W, uint16_t* __restrict__ out,
                                                          size_t ngrp, int K) {
    const size_t gi = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (gi >= ngrp) return;
    const int nb = K >> 8;
    const size_t blkg = gi >> 4;                       // global block index (row * nb + b)
    const int grp = (int)(gi & 15);                    // 16-weight group within the block
    const size_t row = blkg / nb;
    const int b = (int)(blkg - row * nb);
    const uint8_t *ql, *qh, *sc, *dp;
    if constexpr (F == QMM_Q6_K) {
        const uint8_t* bp = W + blkg * 210;
        ql = bp; qh = bp + 128; sc = bp + 192; dp = bp + 208;
    } else {
        const uint8_t* rp = W + row * ((size_t)nb * 210);
        ql = rp + (size_t)b * 128; qh = rp + (size_t)nb * 128 + (size_t)b * 64;
        sc = rp + (size_t)nb * 192 + (size_t)b * 16; dp = rp + (size_t)nb * 208 + (size_t)b * 2;
    }
    const float d = h2f((uint32_t)dp[0] | ((uint32_t)dp[1] << 8));
    // element e = 16 * grp + i: half n = e / 128, r = e % 128, quarter g = r / 32, l = r % 32
    const int e0 = 16 * grp, n = e0 >> 7, r0 = e0 & 127, g = r0 >> 5, l0 = r0 & 31;
    const float ds = d * (float)(int8_t)sc[8 * n + (l0 >> 4) + 2 * g];
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
        uint32_t bf[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int l = l0 + i + k;
            const uint32_t lo = ql[64 * n + l + 32 * (g & 1)], hi = qh[32 * n + l];
            const int q = (int)((g < 2 ? (lo & 15u) : (lo >> 4)) | (((hi >> (2 * g)) & 3u) << 4)) - 32;
            bf[k] = f2bf_bits(ds * (float)q);
        }
        o[i >> 1] = bf[0] | (bf[1] << 16);
    }
    uint4* dst = (uint4*)(out + row * (size_t)K + (size_t)b * 256 + e0);
    dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
    dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
}

#pragma clang fp contract(on)

// ------------------------------------------------------------------------------------------
// bf16 <-> f32 helpers (gemm.hip:77-95 semantics; bf16 from f32 by RNE without a NaN case)
__global__ void k_f32_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ o, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) o[i] = (uint16_t)f2bf_bits(x[i]);
}
__global__ void k_bf16_to_f32(const uint16_t* __restrict__ x, float* __restrict__ o, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) o[i] = bf2f(x[i]);
}
// rows m < M of a [M][Nt] bf16 matrix, columns off..off+N (plus a second matrix when x2) -> f32 [M][N]
__global__ void k_bf16_to_f32_seg2(const uint16_t* __restrict__ x, const uint16_t* __restrict__ x2, int Nt, int off, int N,
                                   float* __restrict__ o, int M) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)M * N) return;
    const int m = (int)(i / N), c = (int)(i % N);
    const size_t idx = (size_t)m * Nt + off + c;
    float v = bf2f(x[idx]);
    if (x2) v += bf2f(x2[idx]);
    o[i] = v;
}

// ------------------------------------------------------------------------------------------
// Tile choice of the dequantising GEMM (gemm_tile.hpp).  Every tile runs the same chain of matrix instructions over K, so the
// choice changes no bit: it may look at everything.  The busiest of the CUs gets q = ceil(tiles / CUs) workgroups, and a
// step of 64 takes it about kStep[format][tile].first ns for one of them and .more for each further one (measured on 256
// CUs with 256 q tiles, q = 1 .. 3, K = 2048 and 8192; two or three workgroups of the small tiles share a CU and hide
// each other's waits).  The large tiles do the most work per ns (192 x 256: 37 blocks of 32 x 32 per us, 16 x 16 by
// producers: 3 to 10), the small ones fill the chip where M x N is small: 40 x 1024 x 5120 in 9 us against 38 with
// 64 x 128, 2048 x 17408 x 5120 in 316 us against 1050 with 64 x 64 by producers.
struct TileShape { int bm, bn, fixed, more; };       // rows, columns; ns for the launch, first loads and stores, the same for each further workgroup
constexpr TileShape kTiles[] = {{16, 16, 4000, 0},      {32, 16, 3200, 1400},   {64, 16, 3400, 2400},   {48, 32, 4500, 1500},   {64, 32, 4700, 1600},
                                {64, 64, 2600, 900},    {128, 64, 4500, 1800},  {64, 128, 2500, 3800},  {96, 128, 6100, 1800},  {128, 128, 7900, 1800},
                                {160, 128, 8100, 2100}, {192, 128, 10500, 4700}, {128, 256, 8500, 4800}, {192, 256, 10900, 8000}, {256, 256, 13200, 9200}};
constexpr int kNumTiles = (int)(sizeof(kTiles) / sizeof(kTiles[0]));
struct StepNs { uint16_t first, more; };
constexpr StepNs kStep[7][kNumTiles] = {
    {{77, 74}, {104, 104}, {137, 131}, {161, 207}, {178, 228}, {360, 357}, {429, 430}, {463, 318}, {496, 398}, {540, 484}, {630, 573}, {695, 721}, {931, 944}, {1278, 1243}, {1644, 1628}},   // Q4_K
    {{103, 99}, {126, 130}, {161, 177}, {207, 243}, {226, 284}, {452, 441}, {523, 508}, {525, 369}, {537, 489}, {662, 545}, {716, 637}, {771, 842}, {1090, 1145}, {1405, 1389}, {1726, 1695}},   // Q5_K
    {{99, 75}, {125, 128}, {163, 159}, {185, 210}, {204, 231}, {336, 330}, {421, 411}, {555, 445}, {627, 485}, {711, 587}, {756, 668}, {843, 847}, {1143, 1210}, {1453, 1461}, {1768, 1772}},   // IQ4_XS
    {{141, 40}, {148, 119}, {172, 175}, {164, 204}, {177, 216}, {361, 347}, {423, 413}, {628, 460}, {704, 505}, {752, 582}, {802, 657}, {888, 848}, {1173, 1207}, {1468, 1498}, {1810, 1747}},   // Q6_K
    {{87, 90}, {112, 141}, {147, 181}, {211, 207}, {232, 226}, {390, 372}, {464, 440}, {550, 474}, {607, 517}, {642, 594}, {684, 676}, {788, 832}, {1096, 1131}, {1382, 1399}, {1672, 1674}},   // Q8_0
    {{109, 87}, {130, 143}, {166, 175}, {191, 239}, {210, 255}, {395, 371}, {462, 453}, {608, 439}, {686, 525}, {776, 578}, {813, 671}, {876, 853}, {1236, 1234}, {1472, 1515}, {1780, 1755}},   // Q5_1
    {{74, 88}, {103, 113}, {166, 168}, {202, 185}, {224, 211}, {352, 339}, {442, 442}, {612, 591}, {666, 664}, {727, 736}, {815, 824}, {918, 868}, {1336, 1223}, {1521, 1537}, {1732, 1727}},   // bf16
};
constexpr int step_row(int f) { return f == QMM_W_BF16 ? 6 : f; }
static_assert(QMM_Q4_K == 0 && QMM_Q5_K == 1 && QMM_IQ4_XS == 2 && QMM_Q6_K_SOA == 3 && QMM_Q8_0_SOA == 4 && QMM_Q5_1_SOA == 5, "");

int tile_count(const TileShape& t, int M, int N) { return ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn); }

// the operands' span in a tile must fit a buffer resource (32-bit offsets)
bool tile_fits(const TileShape& t, const GemmArgs& a) {
    const size_t ra = (size_t)std::min(a.M, t.bm) - 1, rw = (size_t)std::min(a.N, t.bn) - 1;
    return ra * a.lda + (size_t)a.K * 2 <= 0xffffffffu && rw * a.ldw + a.rowbytes <= 0xffffffffu;
}

int pick_tile(int f, const GemmArgs& a) {
    int best = -1;
    long long cost = 0;
    const int cus = device_cu_count(), nk = a.K / 64;
    for (int i = 0; i < kNumTiles; ++i) {
        const TileShape& t = kTiles[i];
        if (!tile_fits(t, a)) continue;
        const StepNs& st = kStep[step_row(f)][i];
        const long long q = (tile_count(t, a.M, a.N) + cus - 1) / cus;
        const long long c = nk * (st.first + (q - 1) * st.more) + t.fixed + (q - 1) * t.more;
        if (best < 0 || c < cost) { best = i; cost = c; }
    }
    return best;
}

template <int F, bool OUT_BF16, int NRB, int CW>
int launch_tile(const GemmArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((k_gemm_tile<F, NRB, CW, OUT_BF16>), dim3(tile_count({32 * NRB, 32 * CW, 0, 0}, a.M, a.N)), dim3(64 * CW), 0, s, a);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}
template <int F, bool OUT_BF16, int R, int CB, int CR, int CC, int B>
int launch_few(const GemmArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((k_gemm_few<F, R, CB, CR, CC, B, OUT_BF16>), dim3(tile_count({16 * R, 16 * CB, 0, 0}, a.M, a.N)),
                       dim3(64 * gf_waves<F, R, CB, CR, CC, B>), 0, s, a);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

// D = A . W^T with W from source F, f32 or bf16 (RNE) out; K % 64 == 0
template <int F, bool OUT_BF16>
int launch_gemm(GemmArgs a, hipStream_t s) {
    const int tile = pick_tile(F, a);
    if (tile < 0) {
        // rows so far apart that no tile's fit a buffer resource (strides above 138 million elements): as many rows and
        // columns at a time as do, down to one of each
        auto most = [](int n, size_t ld, size_t row) { return row > 0xffffffffu ? 0 : (int)std::min<size_t>(n, (0xffffffffu - row) / ld + 1); };
        const int m = most(a.M, a.lda, (size_t)a.K * 2), n = most(a.N, a.ldw, a.rowbytes);
        if (m == 0 || n == 0) return QMM_ERR_SHAPE;
        for (int m0 = 0; m0 < a.M; m0 += m)
            for (int n0 = 0; n0 < a.N; n0 += n) {
                GemmArgs p = a;
                p.A += (size_t)m0 * a.lda;
                p.W += (size_t)n0 * a.ldw;
                p.D = (uint8_t*)a.D + ((size_t)m0 * a.ldd + n0) * (OUT_BF16 ? 2 : 4);
                p.M = std::min(m, a.M - m0);
                p.N = std::min(n, a.N - n0);
                if (int e = launch_gemm<F, OUT_BF16>(p, s)) return e;
            }
        return QMM_OK;
    }
    // rows past M and N read at an offset that is out of the tile's range (and stays so with a row's bytes added), or at
    // row 0 where the range leaves no such offset
    const TileShape& t = kTiles[tile];
    auto past = [](size_t rows, size_t ld, size_t row) {
        const size_t span = (rows - 1) * ld + row;
        return span + row <= 0xffffff00u ? (uint32_t)(0xffffff00u - row) : 0u;
    };
    a.apast = past((size_t)std::min(a.M, t.bm), a.lda, (size_t)a.K * 2);
    a.wpast = past((size_t)std::min(a.N, t.bn), a.ldw, a.rowbytes);
    switch (tile) {
        case 0: return launch_few<F, OUT_BF16, 1, 1, 1, 1, 4>(a, s);
        case 1: return launch_few<F, OUT_BF16, 2, 1, 2, 1, 4>(a, s);
        case 2: return launch_few<F, OUT_BF16, 4, 1, 2, 1, 4>(a, s);
        case 3: return launch_few<F, OUT_BF16, 3, 2, 3, 1, 4>(a, s);
        case 4: return launch_few<F, OUT_BF16, 4, 2, 2, 2, 4>(a, s);
        case 5: return launch_few<F, OUT_BF16, 4, 4, 2, 2, 2>(a, s);
        case 6: return launch_few<F, OUT_BF16, 8, 4, 4, 2, 2>(a, s);
        case 7: return launch_tile<F, OUT_BF16, 2, 4>(a, s);
        case 8: return launch_tile<F, OUT_BF16, 3, 4>(a, s);
        case 9: return launch_tile<F, OUT_BF16, 4, 4>(a, s);
        case 10: return launch_tile<F, OUT_BF16, 5, 4>(a, s);
        case 11: return launch_tile<F, OUT_BF16, 6, 4>(a, s);
        case 12: return launch_tile<F, OUT_BF16, 4, 8>(a, s);
        case 13: return launch_tile<F, OUT_BF16, 6, 8>(a, s);
        default: return launch_tile<F, OUT_BF16, 8, 8>(a, s);
    }
}


// ---- bf16 dequantisation of the other formats (gemm.hip:16-50,83-92 of the reference): one thread
// per 32-weight sub-block (dq_sub32: exact f32), 64 bytes of bf16 out, round-to-nearest-even
// (gemm.hip:12).
template <int F>
__global__ void __launch_bounds__(256) k_dequant_fmt_bf16(const uint8_t* __restrict__ W, uint16_t* __restrict__ out,
                                                         size_t nsub, int K) {
    const size_t g = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= nsub) return;
    const int n32 = K >> 5;
    const size_t row = g / n32;
    const int sb = (int)(g - row * n32);
    float w[32];
    dq_sub32<F>(W + row * fmt_row_bytes_rt(F, K), K, sb, w);
    uint4* dst = (uint4*)(out + row * (size_t)K + 32 * (size_t)sb);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = f2bf_bits(w[8 * v + 2 * k]) | (f2bf_bits(w[8 * v + 2 * k + 1]) << 16);
        dst[v] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

}  // namespace
}  // namespace qmm

using namespace qmm;

extern "C" {

int qmm_dequant_bf16(int fmt, const void* W, uint16_t* out, int N, int K, void* stream) {
    if (!W || !out) return QMM_ERR_NULL;
    // K % 256, or K % 64 (Q8_0_SOA) / K % 32 (Q5_1_SOA) for the row-SoA repacks of 32-weight blocks
    const int kg = fmt == QMM_Q5_1_SOA ? 32 : fmt == QMM_Q8_0_SOA ? 64 : 256;
    if (N <= 0 || K <= 0 || K % kg != 0) return QMM_ERR_SHAPE;
    hipStream_t s = (hipStream_t)stream;
    const size_t nb = (size_t)N * (K / 256);
    const size_t nsub = (size_t)N * (K / 32);      // 32-weight sub-blocks
    switch (fmt) {
        case QMM_Q4_K:
            hipLaunchKernelGGL(k_dequant_q4k_bf16, dim3((unsigned)((nb * 8 + 255) / 256)), dim3(256), 0, s, (const uint8_t*)W, out,
                               nb * 8, K);
            break;
        case QMM_Q6_K:
            hipLaunchKernelGGL(k_dequant_q6k_bf16<QMM_Q6_K>, dim3((unsigned)((nb * 16 + 255) / 256)), dim3(256), 0, s,
                               (const uint8_t*)W, out, nb * 16, K);
            break;
        case QMM_Q6_K_SOA:
            hipLaunchKernelGGL(k_dequant_q6k_bf16<QMM_Q6_K_SOA>, dim3((unsigned)((nb * 16 + 255) / 256)), dim3(256), 0, s,
                               (const uint8_t*)W, out, nb * 16, K);
            break;
#define QMM_DQF(F) case F: hipLaunchKernelGGL(k_dequant_fmt_bf16<F>, dim3((unsigned)((nsub + 255) / 256)), dim3(256), 0, s, \
                                              (const uint8_t*)W, out, nsub, K); break;
        QMM_DQF(QMM_Q5_K) QMM_DQF(QMM_IQ4_XS) QMM_DQF(QMM_Q8_0_SOA) QMM_DQF(QMM_Q5_1_SOA)
#undef QMM_DQF
        default: return QMM_ERR_FORMAT;
    }
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

int qmm_gemm_wq(int fmt, const void* W, const uint16_t* A, float* D, int M, int N, int K, void* stream) {
    if (!(fmt == QMM_Q4_K || fmt == QMM_Q5_K || fmt == QMM_IQ4_XS || fmt == QMM_Q6_K_SOA || fmt == QMM_Q8_0_SOA ||
          fmt == QMM_Q5_1_SOA))
        return QMM_ERR_FORMAT;
    if (!W || !A || !D) return QMM_ERR_NULL;
    // K % 256 for the block formats (K % 512 for Q6_K_SOA: an even block count keeps its streams dword
    // aligned), K % 128 for the 32-weight SoA formats
    const int kg = (fmt == QMM_Q8_0_SOA || fmt == QMM_Q5_1_SOA) ? 128 : fmt == QMM_Q6_K_SOA ? 512 : 256;
    if (M <= 0 || N <= 0 || K <= 0 || K % kg != 0) return QMM_ERR_SHAPE;
    const size_t rb = fmt_row_bytes_rt(fmt, K);
    const GemmArgs a{(const uint8_t*)A, (const uint8_t*)W, D, (uint32_t)K * 2u, (uint32_t)rb, (uint32_t)rb, M, N, K, N, 0, 0};
    hipStream_t s = (hipStream_t)stream;
    switch (fmt) {
        case QMM_Q4_K: return launch_gemm<QMM_Q4_K, false>(a, s);
        case QMM_Q5_K: return launch_gemm<QMM_Q5_K, false>(a, s);
        case QMM_IQ4_XS: return launch_gemm<QMM_IQ4_XS, false>(a, s);
        case QMM_Q6_K_SOA: return launch_gemm<QMM_Q6_K_SOA, false>(a, s);
        case QMM_Q8_0_SOA: return launch_gemm<QMM_Q8_0_SOA, false>(a, s);
        default: return launch_gemm<QMM_Q5_1_SOA, false>(a, s);
    }
}

int qmm_gemm_bf16_ld(const uint16_t* A, int lda, const uint16_t* W, int ldw, uint16_t* D, int M, int N, int K, void* stream) {
    if (!A || !W || !D) return QMM_ERR_NULL;
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || lda < K || ldw < K) return QMM_ERR_SHAPE;
    // 16-byte row pieces: both operands' rows start 16-byte aligned
    if (((uintptr_t)A | (uintptr_t)W) % 16 != 0 || lda % 8 != 0 || ldw % 8 != 0) return QMM_ERR_ARG;
    // the limit of the call since its first kernel, which addressed A with 32-bit element offsets; nothing needs it now
    if ((uint64_t)(M - 1) * (uint64_t)lda + (uint64_t)K > 0xffffffffull) return QMM_ERR_SHAPE;
    return launch_gemm<QMM_W_BF16, true>(GemmArgs{(const uint8_t*)A, (const uint8_t*)W, D, (uint32_t)lda * 2u, (uint32_t)ldw * 2u, (uint32_t)K * 2u,
                                                  M, N, K, N, 0, 0}, (hipStream_t)stream);
}

int qmm_gemm_tile(int fmt, int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || fmt == QMM_Q6_K || fmt > QMM_Q5_1_SOA) return QMM_ERR_ARG;
    const int f = fmt < 0 ? QMM_W_BF16 : fmt;
    const uint32_t rb = fmt < 0 ? (uint32_t)K * 2u : (uint32_t)fmt_row_bytes_rt(fmt, K);
    return pick_tile(f, GemmArgs{nullptr, nullptr, nullptr, (uint32_t)K * 2u, rb, rb, M, N, K, N, 0, 0});
}

int qmm_gemm_bf16(const uint16_t* A, const uint16_t* W, uint16_t* D, int M, int N, int K, void* stream) {
    return qmm_gemm_bf16_ld(A, K, W, K, D, M, N, K, stream);
}

int qmm_f32_to_bf16(const float* x, uint16_t* out, size_t n, void* stream) {
    if (!x || !out) return QMM_ERR_NULL;
    if (n == 0) return QMM_OK;
    hipLaunchKernelGGL(k_f32_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, out, n);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

int qmm_bf16_to_f32(const uint16_t* x, float* out, size_t n, void* stream) {
    if (!x || !out) return QMM_ERR_NULL;
    if (n == 0) return QMM_OK;
    hipLaunchKernelGGL(k_bf16_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, out, n);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

int qmm_bf16_to_f32_seg2(const uint16_t* x, const uint16_t* x2, int Nt, int off, int N, float* out, int M, void* stream) {
    if (!x || !out) return QMM_ERR_NULL;
    if (M < 0 || N < 0 || off < 0 || off + N > Nt) return QMM_ERR_SHAPE;
    const size_t n = (size_t)M * N;
    if (n == 0) return QMM_OK;
    hipLaunchKernelGGL(k_bf16_to_f32_seg2, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, x2, Nt, off,
                       N, out, M);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

int qmm_bf16_to_f32_seg(const uint16_t* x, int Nt, int off, int N, float* out, int M, void* stream) {
    return qmm_bf16_to_f32_seg2(x, nullptr, Nt, off, N, out, M, stream);
}

}  // extern "C"
