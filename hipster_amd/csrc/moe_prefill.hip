// moe_prefill.hip -- MoE prefill on gfx950: device-side expert sort (histogram, prefix scan, stable
// scatter, tiles), the grouped expert GEMM over the sorted rows for Q4_K rows of one or two blocks (other
// rows and formats: moe_gemm_fmt.hip), and silu(g)*u -> bf16.
//
// Entry points (C ABI, include/hipster_qmm.h) and what they replace in the reference:
//   qmm_moe_sort        the host path of engine/src/qwen4exp.cpp:628-645 (blocking device->host
//                       copy of the ids, std::sort by (expert, slot), tile building, three
//                       host->device copies) -- here one workgroup on the device, no host sync
//   qmm_moe_gemm_bf16   moe_gemm (engine/kernels/gemv.h:49-50, gemv.hip:909-969,1377-1381) with
//                       bf16 activations; the tile count is read on the device
//   qmm_moe_gemm_gate_up_bf16  the gate and up moe_gemm calls plus moe_silu_quant of
//                       qwen4exp.cpp:646-648 in one launch, writing h = bf16(silu(g) * u)
//   qmm_moe_silu_bf16   moe_silu_quant (fn.hip:206-211) for the bf16 path: h = bf16(silu(g) * u)
#include "qmm_common.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace qmm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ------------------------------------------------------------------------------------------
// Expert sort.  Slots te = t*nslot + e are ordered by key = id + 1 (0 = shared expert, id -1, then
// the experts ascending), stable in te: the reference's std::sort by (expert id, te)
// (qwen4exp.cpp:631-632).  A workgroup of 16 waves; wave w owns a contiguous slot range.  Pass 1
// counts keys per wave; pass 2 turns the counts into per-(key, wave) start offsets, key-major then
// wave order; pass 3 scatters each wave's range in order, a lane's rank among equal keys of its
// 64-slot chunk coming from ballot peer masks over the key bits -- deterministic and stable.  Large
// slot counts spread the same passes over several workgroups (k_moe_sort_count / _offsets /
// _scatter); small ones run in one (k_moe_sort).
// Tiles: per key, ceil(count / maxc) tiles of consecutive sorted positions (the reference cuts a
// tile at each expert change and every maxc positions, qwen4exp.cpp:636-641); routed-expert tiles
// first in expert order, then the shared-expert tiles.  counts = {routed tiles, shared tiles}.
constexpr int kSortThreads = 1024, kSortWaves = kSortThreads / 64, kMaxKeys = 1025, kSortBatch = 16, kSortMaxGroups = 64;

// exclusive scan over the workgroup of one int per thread; *total gets the sum
__device__ __forceinline__ int block_exscan(int v, int* wsum, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(x, o, 64);
        if (lane >= o) x += u;
    }
    __syncthreads();
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    if (wave == 0) {
        int y = lane < kSortWaves ? wsum[lane] : 0;
#pragma unroll
        for (int o = 1; o < kSortWaves; o <<= 1) {
            const int u = __shfl_up(y, o, 64);
            if (lane >= o) y += u;
        }
        if (lane < kSortWaves) wsum[lane] = y;
    }
    __syncthreads();
    *total = wsum[kSortWaves - 1];
    return x - v + (wave > 0 ? wsum[wave - 1] : 0);
}

// Slots [lo, hi) of one workgroup are split over its 16 waves in contiguous runs of `per` (a
// multiple of 64); the same split is used by every kernel that counts or scatters them.
__device__ __forceinline__ void wave_range(int lo, int hi, int wave, int& wlo, int& whi) {
    const int per = ((hi - lo + kSortWaves - 1) / kSortWaves + 63) & ~63;
    wlo = min(hi, lo + wave * per);
    whi = min(hi, wlo + per);
}

// the sort key of an id: id + 1 (0 = the shared expert), ids outside [-1, nkeys - 2] clamped into
// that range, so a bad router output sorts wrongly but never indexes outside the count tables
__device__ __forceinline__ int sort_key(int id, int nkeys) { return min(max(id + 1, 0), nkeys - 1); }

// pass 1: key counts of the wave's slots into cnt[wave * nkeys + key] (LDS, zeroed by the caller).
// The ids are
// loaded kSortBatch per lane at a time, so the loads overlap instead of each waiting behind the
// previous LDS atomic.
__device__ __forceinline__ void sort_count(const int* __restrict__ ids, int lo, int hi, int nkeys, int* cnt) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int c0 = lo; c0 < hi; c0 += 64 * kSortBatch) {
        int kk[kSortBatch];
#pragma unroll
        for (int u = 0; u < kSortBatch; ++u) {      // unconditional (clamped) loads: no wait per load
            const int i = c0 + 64 * u + lane;
            const int v = sort_key(ids[min(i, hi - 1)], nkeys);
            kk[u] = i < hi ? v : -1;
        }
#pragma unroll
        for (int u = 0; u < kSortBatch; ++u)
            if (kk[u] >= 0) atomicAdd(&cnt[wave * nkeys + kk[u]], 1);
    }
}

// pass 3: stable scatter of the wave's slots in order; cnt[wave * nkeys + key] holds the wave's
// running offset of each key.  A lane's rank among the equal keys of its 64-slot chunk comes from
// ballot peer masks over the 11 key bits.
__device__ __forceinline__ void sort_scatter(const int* __restrict__ ids, int lo, int hi, int nkeys, int* cnt,
                                             int* __restrict__ kpos) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long lt = (1ull << lane) - 1ull;
    for (int b0 = lo; b0 < hi; b0 += 64 * kSortBatch) {
        int kk[kSortBatch];
#pragma unroll
        for (int u = 0; u < kSortBatch; ++u) {
            const int i = b0 + 64 * u + lane;
            const int v = sort_key(ids[min(i, hi - 1)], nkeys);
            kk[u] = i < hi ? v : 0;
        }
#pragma unroll
        for (int u = 0; u < kSortBatch; ++u) {
            const int c0 = b0 + 64 * u;
            if (c0 >= hi) break;
            const int i = c0 + lane;
            const bool valid = i < hi;
            const int key = kk[u];
            unsigned long long peers = __ballot(valid);
            for (int b = 0; b < 11; ++b) {
                const bool bit = (key >> b) & 1;
                const unsigned long long m = __ballot(bit);
                peers &= bit ? m : ~m;
            }
            const int rank = __popcll(peers & lt);
            int pos = 0;
            if (valid) pos = cnt[wave * nkeys + key] + rank;
            __builtin_amdgcn_wave_barrier();
            if (valid) {
                kpos[i] = pos;
                if (rank == 0) cnt[wave * nkeys + key] += __popcll(peers);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// tiles of the keys [k0, k1) owned by this thread, given each key's start and count (routed
// experts, keys >= 1, first in key order; then thread 0 writes the shared expert's, key 0)
__device__ __forceinline__ void sort_tiles(const int* start, const int* tot, int k0, int k1, int maxc, int* wsum,
                                           qmm_moe_tile* __restrict__ tiles, int* __restrict__ counts) {
    int nt = 0;
    for (int k = max(k0, 1); k < k1; ++k) nt += (tot[k] + maxc - 1) / maxc;
    int nrouted = 0;
    int tb = block_exscan(nt, wsum, &nrouted);
    for (int k = max(k0, 1); k < k1; ++k) {
        for (int r = 0; r < tot[k]; r += maxc) {
            qmm_moe_tile tl;
            tl.expert = k - 1; tl.k0 = start[k] + r; tl.ncols = min(maxc, tot[k] - r);
            tiles[tb++] = tl;
        }
    }
    if (threadIdx.x == 0) {
        int n = 0;
        for (int r = 0; r < tot[0]; r += maxc) {
            qmm_moe_tile tl;
            tl.expert = -1; tl.k0 = start[0] + r; tl.ncols = min(maxc, tot[0] - r);
            tiles[nrouted + n++] = tl;
        }
        counts[0] = nrouted;
        counts[1] = n;
    }
}

// Whole sort in one workgroup (small slot counts)
__global__ void __launch_bounds__(kSortThreads) k_moe_sort(const int* __restrict__ ids, int ns, int nslot, int nkeys, int maxc,
                                                           int* __restrict__ kpos, qmm_moe_tile* __restrict__ tiles,
                                                           int* __restrict__ counts) {
    extern __shared__ int sm[];
    int* cnt = sm;                                   // [kSortWaves][nkeys]: per-wave counts, then running offsets
    int* tot = cnt + kSortWaves * nkeys;             // [nkeys]
    int* start = tot + nkeys;                        // [nkeys]
    __shared__ int wsum[kSortWaves];
    const int tid = threadIdx.x, wave = tid >> 6;
    for (int i = tid; i < kSortWaves * nkeys; i += kSortThreads) cnt[i] = 0;
    __syncthreads();
    int lo, hi;
    wave_range(0, ns, wave, lo, hi);
    sort_count(ids, lo, hi, nkeys, cnt);
    __syncthreads();
    // each thread owns a contiguous key range [k0, k1)
    const int kper = (nkeys + kSortThreads - 1) / kSortThreads;
    const int k0 = min(nkeys, tid * kper), k1 = min(nkeys, k0 + kper);
    int run = 0;
    for (int k = k0; k < k1; ++k) {
        int s = 0;
        for (int w = 0; w < kSortWaves; ++w) s += cnt[w * nkeys + k];
        tot[k] = s;
        run += s;
    }
    int total = 0;
    int base = block_exscan(run, wsum, &total);
    // pass 2: per-(key, wave) start offsets
    for (int k = k0; k < k1; ++k) {
        start[k] = base;
        for (int w = 0; w < kSortWaves; ++w) {
            const int c = cnt[w * nkeys + k];
            cnt[w * nkeys + k] = base;
            base += c;
        }
    }
    __syncthreads();
    sort_scatter(ids, lo, hi, nkeys, cnt, kpos);
    sort_tiles(start, tot, k0, k1, maxc, wsum, tiles, counts);
}

// The same sort over G workgroups (large slot counts), in two launches: each workgroup counts the
// keys of its contiguous slot range into hist[g][key] (global scratch); then each workgroup counts
// its range again per wave, derives its start per (key, wave) from the whole table (keys before,
// then the same key in earlier workgroups and waves) and scatters; workgroup 0 also writes the
// tiles.  The order is the one-workgroup order: key, then workgroup, then wave, then slot -- i.e.
// key, then slot.
__global__ void __launch_bounds__(kSortThreads) k_moe_sort_count(const int* __restrict__ ids, int ns, int nkeys, int per,
                                                                 int* __restrict__ hist) {
    extern __shared__ int sm[];
    const int tid = threadIdx.x, wave = tid >> 6;
    for (int i = tid; i < kSortWaves * nkeys; i += kSortThreads) sm[i] = 0;
    __syncthreads();
    const int glo = min(ns, (int)blockIdx.x * per), ghi = min(ns, glo + per);
    int lo, hi;
    wave_range(glo, ghi, wave, lo, hi);
    sort_count(ids, lo, hi, nkeys, sm);
    __syncthreads();
    for (int k = tid; k < nkeys; k += kSortThreads) {
        int s = 0;
        for (int w = 0; w < kSortWaves; ++w) s += sm[w * nkeys + k];
        hist[(size_t)blockIdx.x * nkeys + k] = s;
    }
}

__global__ void __launch_bounds__(kSortThreads) k_moe_sort_scatter(const int* __restrict__ ids, int ns, int nkeys, int per, int G,
                                                                   int maxc, const int* __restrict__ hist, int* __restrict__ kpos,
                                                                   qmm_moe_tile* __restrict__ tiles, int* __restrict__ counts) {
    extern __shared__ int sm[];
    int* cnt = sm;                                   // [kSortWaves][nkeys]
    int* tot = cnt + kSortWaves * nkeys;             // [nkeys]
    int* start = tot + nkeys;                        // [nkeys]
    __shared__ int wsum[kSortWaves];
    const int tid = threadIdx.x, wave = tid >> 6, g = blockIdx.x;
    for (int i = tid; i < kSortWaves * nkeys; i += kSortThreads) cnt[i] = 0;
    __syncthreads();
    const int glo = min(ns, g * per), ghi = min(ns, glo + per);
    int lo, hi;
    wave_range(glo, ghi, wave, lo, hi);
    sort_count(ids, lo, hi, nkeys, cnt);
    // this workgroup's start per key: the keys before it, then the same key in earlier workgroups
    const int kper = (nkeys + kSortThreads - 1) / kSortThreads;
    const int k0 = min(nkeys, tid * kper), k1 = min(nkeys, k0 + kper);
    int run = 0;
    for (int k = k0; k < k1; ++k) {
        int s = 0, before = 0;
        for (int gg = 0; gg < G; ++gg) {
            const int c = hist[(size_t)gg * nkeys + k];
            before += gg < g ? c : 0;
            s += c;
        }
        tot[k] = s;
        start[k] = before;                           // offset within the key for now
        run += s;
    }
    int total = 0;
    int base = block_exscan(run, wsum, &total);      // also orders the count pass before the reads below
    for (int k = k0; k < k1; ++k) {
        int r = base + start[k];
        start[k] = base;
        base += tot[k];
        for (int w = 0; w < kSortWaves; ++w) {
            const int c = cnt[w * nkeys + k];
            cnt[w * nkeys + k] = r;
            r += c;
        }
    }
    __syncthreads();
    sort_scatter(ids, lo, hi, nkeys, cnt, kpos);
    if (g == 0) sort_tiles(start, tot, k0, k1, maxc, wsum, tiles, counts);
}

// rowtok[kpos[i]] = token of slot i: the inverse permutation, written by the whole grid (scattered
// 4-byte stores issued from the one sorting workgroup would all queue on a single CU)
__global__ void __launch_bounds__(256) k_moe_rowtok(const int* __restrict__ kpos, int* __restrict__ rowtok, int ns, int nslot) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < ns && (unsigned)kpos[i] < (unsigned)ns) rowtok[kpos[i]] = i / nslot;
}

// ------------------------------------------------------------------------------------------
// Grouped expert GEMM for rows of one or two Q4_K blocks.  A tile holds up to 128 sorted rows:
// D[k0 + r][n] = sum_k A[row(r)][k] * W_e[n][k] for r < ncols, row(r) = rowtab[k0 + r] (or k0 + r), W_e the
// expert's Q4_K matrix (the shared matrix when expert < 0).
constexpr int XBM = 128, XBW = 256;                         // rows of a tile, weight rows of a block

struct XArgs {
    const uint8_t* w0;     // expert matrices, expert e at w0 + e * ebytes
    const uint8_t* w0sh;   // shared-expert matrix
    size_t ebytes;
    const qmm_moe_tile* tiles;
    const int* counts;
    const int* rowtab;
    const uint16_t* A;
    void* D;               // f32 [k][ldd]
    int N, nb;             // nb = 256-row weight blocks per tile
    int ldd;               // row stride of D (elements)
    int cap;               // capacity of tiles (the device count is clamped to it)
    int bpu;               // weight blocks per work unit
};

// scales of K step j (qs pair j: sub-blocks 2j, 2j+1) of a Q4_K block header, pre-scaled for
// q4_bf16x8_mix: {d*sc[2j] * 2^24, dmin*m[2j], d*sc[2j+1] * 2^20, dmin*m[2j+1]}
struct StepScl { float sa, ma, sb, mb; };
__device__ __forceinline__ StepScl q4k_step_scales(const uint4 hd, int j) {
    const float d = h2f(hd.x), dmin = h2f(hd.x >> 16);
    const Q4kScaleBytes sb = q4k_scale_bytes(hd.y, hd.z, hd.w);
    StepScl c;
    c.sa = d * (float)byte8(sb.sc_lo, sb.sc_hi, 2 * j) * 16777216.f;
    c.ma = dmin * (float)byte8(sb.m_lo, sb.m_hi, 2 * j);
    c.sb = d * (float)byte8(sb.sc_lo, sb.sc_hi, 2 * j + 1) * 1048576.f;
    c.mb = dmin * (float)byte8(sb.m_lo, sb.m_hi, 2 * j + 1);
    return c;
}

// The tile's activations are resident in LDS: K = 256 KB, KB = 2 (the MoE down projection) or 1.  Work unit = (tile, run
// of bpu consecutive 256-row weight blocks).  The tile's A rows (at most 128 x 512 bf16 = 128 KiB) are copied global -> LDS once per unit; after that every wave
// works alone: it streams its own 32 weight rows of each block straight into registers, dequantises
// them and multiplies them against A fragments read from LDS, block after block, and stores each
// block's f32 results.  The main loop has no workgroup barrier and no LDS writes, and A is read from
// global memory once per unit instead of once per weight block.
// The K order is the tile core's (same MFMA sequence, so the same results bit for bit): per 64-wide
// K step lane l (weight row l%32, h = l/32) takes qs bytes 16h..16h+15 of the step's pair in one load (as
// two 8-byte pieces it cost the address units twice the instructions: 112 -> 106 us at 2048 tokens), slices 0
// and 1 their low nibbles, slices 2 and 3 their high nibbles, and the A fragment of slice s is chunk
// 4 (s / 2) + 2h + s % 2 of the step.  Two weight blocks per unit: 104.8 / 47.3 / 27.2 us at 2048 / 512 / 96 tokens
// against 106.4 / 53.9 / 29.2 with four, whose units were too few for the CUs.  A in LDS: row r at r * (512 KB + 16)
// bytes, so the 16 rows a quarter-wave reads fall in 16 distinct
// bank groups and every fragment address is one lane base plus a constant; one DMA instruction
// copies one row.
constexpr int kAsThreads = 512;
template <int KB>
constexpr int kAsRowBytes = 512 * KB + 16;

// f32 store the compiler does not see (address = wave-uniform base in SGPRs + per-lane 32-bit byte
// offset): its waits for the weight loads issued before it are then computed over loads only (loads
// complete in order, so such a wait can only last longer), instead of the full vmcnt(0) it places
// once loads and stores are both outstanding.  Unlike the DMA helpers it carries no s_nop guard (64
// stores per weight block): its base is only ever advanced by scalar adds, never reloaded by a VALU
// instruction, which tests/test_asm_hazards.py checks on the compiled code.
__device__ __forceinline__ void st_f32_nc(const uint8_t* base, uint32_t voff, float v) {
    asm volatile("global_store_dword %0, %1, %2" : : "v"(voff), "v"(v), "s"(base) : "memory");
}

// one Q4_K block (4 K steps) of the lane's weight row: header and the lane's 16 qs bytes per step j (bytes
// 16h.. of pair j)
struct AsRaw { uint4 hd, q0, q1, q2, q3; };

template <int NRB, int KB>
__device__ __forceinline__ void moe_as_unit(const XArgs& a, const qmm_moe_tile tl, int b0, int b1, const int* rows,
                                            uint8_t* As) {
    const int lane = threadIdx.x & 63, fr = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr uint32_t rowbytes = KB * 144u;
    constexpr int kRow = kAsRowBytes<KB>;
    const int N = a.N;
    const uint8_t* w = tl.expert >= 0 ? a.w0 + (size_t)tl.expert * a.ebytes : a.w0sh;
    if (lane < 32 * KB) {   // A rows 0 .. 32 NRB - 1 -> LDS, one DMA instruction (16 B a lane) per row
        const uint32_t la = lds_addr(As);
        for (int r = wave; r < NRB * 32; r += 8)
            dma16((const uint8_t*)a.A + ((size_t)rows[r] * (256 * KB) + (size_t)(8 * lane)) * 2, la + (uint32_t)(r * kRow));
    }
    // group g = Q4_K block g % KB of weight block b0 + g / KB; the lane's row in it (clamped: rows past
    // N load row N-1 and are not stored)
    const int ng = KB * (b1 - b0);
    auto load = [&](int g, AsRaw& r) {
        const int b = b0 + g / KB;
        const uint8_t* p = w + (size_t)min(b * 256 + 32 * wave + fr, N - 1) * rowbytes + (size_t)(g % KB) * 144;
        const uint8_t* pq = p + 16 + 16 * h;
        r.hd = ld16(p);
        r.q0 = ld16(pq);
        r.q1 = ld16(pq + 32);
        r.q2 = ld16(pq + 64);
        r.q3 = ld16(pq + 96);
    };
    f32x16 acc[NRB];
#pragma unroll
    for (int i = 0; i < NRB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
    AsRaw ra, rb;
    load(0, ra);
    __builtin_amdgcn_s_waitcnt(0);      // the A copy has landed (and group 0)
    __syncthreads();
    // lane bases: row fr (row blocks 0, 1) and row 64 + fr (row blocks 2, 3), chunk 2h
    typedef __attribute__((address_space(3))) const uint8_t lds_u8;
    const lds_u8* alo = (const lds_u8*)As + fr * kRow + 32 * h;
    const lds_u8* ahi = alo + 64 * kRow;
    asm volatile("" : "+v"(ahi));     // a base of its own: otherwise folded into alo + offsets past 64 KiB

    // K step t of the row; the four slices' NRB MFMAs each
    auto step = [&](const uint4 q, const StepScl& c, int t) {
        bf16x8 wv[4];
        wv[0] = q4_bf16x8_mix(q.x, q.y, 0x000f000fu, c.sa, -c.ma);
        wv[1] = q4_bf16x8_mix(q.z, q.w, 0x000f000fu, c.sa, -c.ma);
        wv[2] = q4_bf16x8_mix(q.x, q.y, 0x00f000f0u, c.sb, -c.mb);
        wv[3] = q4_bf16x8_mix(q.z, q.w, 0x00f000f0u, c.sb, -c.mb);
        // A fragments one slice ahead, each slice fenced: two slices' fragments live at most
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        u32x4 af[NRB], an[NRB];
        auto rd = [&](u32x4 (&v)[NRB], int s) {
            const int off = (8 * t + 4 * (s >> 1) + (s & 1)) * 16;
#pragma unroll
            for (int i = 0; i < NRB; ++i)
                v[i] = *(const __attribute__((address_space(3))) u32x4*)((i < 2 ? alo : ahi) + (i & 1) * 32 * kRow + off);
        };
        rd(af, 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) rd(an, s + 1);
#pragma unroll
            for (int i = 0; i < NRB; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[i]), wv[s], acc[i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NRB; ++i) af[i] = an[i];
        }
    };
    // results of weight block b (tile row 32i + 8(e/4) + e%4 + 4h): the uniform row part walks a
    // scalar pointer (kept opaque, so its 64 values are formed one at a time instead of hoisted out of
    // the loop), the lane part (4h rows, column n) is a fixed byte offset; then the set restarts at 0
    auto store = [&](int b) {
        const int n = b * 256 + 32 * wave + fr;
        const uint32_t voff = (uint32_t)(4 * h * a.ldd + n) * 4u;
        int rem = n < N ? tl.ncols - 4 * h : 0;     // the lane stores uniform row offsets below rem
        asm volatile("" : "+v"(rem));               // (compared here, not as 64 hoisted masks)
        const size_t rs = (size_t)a.ldd * 4;
        const uint8_t* p = (const uint8_t*)a.D + (size_t)tl.k0 * rs;
#pragma unroll
        for (int i = 0; i < NRB; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                asm volatile("" : "+s"(p));
                if (32 * i + 8 * (e >> 2) + (e & 3) < rem) st_f32_nc(p, voff, acc[i][e]);
                acc[i][e] = 0.f;
                p += (e & 3) == 3 ? 5 * rs : rs;     // next row: +1, or +5 after the 4th of a group of 8
            }
    };
    // group g (Q4_K block kb of its weight block): the K steps of raw r; the next group's loads go out after
    // the first step, a weight block's results are stored behind its last group.
    // Fenced steps: hoisting a step's A fragments and dequantisation over the previous step's MFMAs
    // runs out of registers.
    auto group = [&](int g, int kb, const AsRaw& r, AsRaw& fill) {
        const int t0 = 4 * kb;
        step(r.q0, q4k_step_scales(r.hd, 0), t0);
        __builtin_amdgcn_sched_barrier(0);
        load(min(g + 1, ng - 1), fill);
        __builtin_amdgcn_sched_barrier(0);
        step(r.q1, q4k_step_scales(r.hd, 1), t0 + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(r.q2, q4k_step_scales(r.hd, 2), t0 + 2);
        __builtin_amdgcn_sched_barrier(0);
        step(r.q3, q4k_step_scales(r.hd, 3), t0 + 3);
        __builtin_amdgcn_sched_barrier(0);
        if (kb == KB - 1) store(b0 + g / KB);
    };
    for (int g = 0; g < ng; g += 2) {
        group(g, 0, ra, rb);
        if (KB == 2 || g + 1 < ng) group(g + 1, KB - 1, rb, ra);
    }
}

// One workgroup per (tile, run of bpu weight blocks); workgroup id i runs on XCD i % 8 and XCD x
// takes tiles x, x+8, ... with all their runs (the runs of a tile share its A rows in one L2).
template <int KB>
__global__ void __launch_bounds__(kAsThreads) k_moe_gemm_as(XArgs a) {
    extern __shared__ __align__(16) uint8_t smem_raw[];
    __shared__ int rows[XBM];
    const int nu = (a.nb + a.bpu - 1) / a.bpu;
    const int id = blockIdx.x, sid = id >> 3;
    const int tix = 8 * (sid / nu) + (id & 7), ui = sid % nu;
    if (tix >= min(a.counts[0] + a.counts[1], a.cap)) return;
    qmm_moe_tile tl = a.tiles[tix];
    tl.ncols = max(1, min(tl.ncols, XBM));
    if (threadIdx.x < XBM) {
        const int k = tl.k0 + min((int)threadIdx.x, tl.ncols - 1);
        rows[threadIdx.x] = a.rowtab ? a.rowtab[k] : k;
    }
    __syncthreads();
    const int b0 = ui * a.bpu, b1 = min(a.nb, b0 + a.bpu);
    switch ((tl.ncols + 31) >> 5) {
        case 1: moe_as_unit<1, KB>(a, tl, b0, b1, rows, smem_raw); break;
        case 2: moe_as_unit<2, KB>(a, tl, b0, b1, rows, smem_raw); break;
        case 3: moe_as_unit<3, KB>(a, tl, b0, b1, rows, smem_raw); break;
        default: moe_as_unit<4, KB>(a, tl, b0, b1, rows, smem_raw); break;
    }
}

template <int KB>
int launch_moe_gemm_as(const XArgs& a, int max_tiles, hipStream_t s) {
    const int nu = (a.nb + a.bpu - 1) / a.bpu;
    const int grid = 8 * ((max_tiles + 7) / 8) * nu;
    hipLaunchKernelGGL(k_moe_gemm_as<KB>, dim3(grid), dim3(kAsThreads), (size_t)XBM * kAsRowBytes<KB>, s, a);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

}  // namespace

namespace {

// ------------------------------------------------------------------------------------------
// h = bf16(silu(g) * u), RNE; silu(x) = x / (1 + __expf(-x)) as the reference (fn.hip:8)
__global__ void __launch_bounds__(256) k_moe_silu_bf16(const float* __restrict__ g, const float* __restrict__ u,
                                                       uint16_t* __restrict__ h, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float x = g[i];
    h[i] = (uint16_t)f2bf_bits(x / (1.f + __expf(-x)) * u[i]);
}

}  // namespace
}  // namespace qmm

using namespace qmm;

extern "C" {

int qmm_moe_sort(const int* ids, int T, int nslot, int nexperts, int maxc, int* kpos, int* rowtok, qmm_moe_tile* tiles,
                 int* counts, void* stream) {
    if (!ids || !kpos || !rowtok || !tiles || !counts) return QMM_ERR_NULL;
    if (T < 0 || nslot < 1 || nexperts < 1 || nexperts + 1 > kMaxKeys || maxc < 1 || maxc > QMM_MOE_MAX_TILE_ROWS) return QMM_ERR_SHAPE;
    const int nkeys = nexperts + 1, ns = T * nslot;
    hipStream_t st = (hipStream_t)stream;
    // G workgroups of at least 1024 slots each, their counts (G x nkeys) held in rowtok until the
    // rowtok kernel overwrites it; one workgroup when that does not give at least 4
    const int G = std::min(std::min(ns / 1024, ns / nkeys), kSortMaxGroups);
    if (G >= 4) {
        const int per = (ns + G - 1) / G;
        const size_t lds_w = (size_t)kSortWaves * nkeys * 4;
        hipLaunchKernelGGL(k_moe_sort_count, dim3(G), dim3(kSortThreads), lds_w, st, ids, ns, nkeys, per, rowtok);
        QMM_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_moe_sort_scatter, dim3(G), dim3(kSortThreads), lds_w + (size_t)2 * nkeys * 4, st, ids, ns, nkeys, per, G,
                           maxc, rowtok, kpos, tiles, counts);
        QMM_LAUNCH_CHECK();
    } else {
        const size_t lds = (size_t)(kSortWaves + 2) * nkeys * 4;
        hipLaunchKernelGGL(k_moe_sort, dim3(1), dim3(kSortThreads), lds, st, ids, ns, nslot, nkeys, maxc, kpos, tiles, counts);
        QMM_LAUNCH_CHECK();
    }
    if (ns > 0) {
        hipLaunchKernelGGL(k_moe_rowtok, dim3((ns + 255) / 256), dim3(256), 0, st, kpos, rowtok, ns, nslot);
        QMM_LAUNCH_CHECK();
    }
    return QMM_OK;
}

int qmm_moe_gemm_bf16(int fmt, int shared_fmt, const void* W, const void* Wsh, size_t ebytes, const qmm_moe_tile* tiles,
                      const int* counts, int max_tiles, const int* rowtab, const uint16_t* A, float* D, int N, int K,
                      void* stream) {
    // the reference's moe_gemm formats (gemv.hip:962-968), routed and shared independent, and IQ4_XS;
    // K granule per format as qmm_gemv_q8 (256; 64 for Q8_0_SOA, 32 for Q5_1_SOA)
    auto fmt_ok = [](int f) { return f == QMM_Q4_K || f == QMM_Q5_K || f == QMM_IQ4_XS || f == QMM_Q8_0_SOA || f == QMM_Q5_1_SOA; };
    auto kgran = [](int f) { return f == QMM_Q5_1_SOA ? 32 : f == QMM_Q8_0_SOA ? 64 : 256; };
    if (!fmt_ok(fmt) || !fmt_ok(shared_fmt)) return QMM_ERR_FORMAT;
    if (!W || !Wsh || !tiles || !counts || !A || !D) return QMM_ERR_NULL;
    if (N <= 0 || K <= 0 || K % kgran(fmt) != 0 || K % kgran(shared_fmt) != 0 || max_tiles < 0) return QMM_ERR_SHAPE;
    if (max_tiles == 0) return QMM_OK;
    // Q4_K (2048 rows, 256 experts, top 8; k_moe_gemm_as against the tile core, us at 96 / 2048 / 4096 tokens): K = 256
    // 11 / 50 / 95 against 16 / 85 / 145, K = 512 17 / 80 / 145 against 21 / 110 / 196: A is read once for two weight blocks and no
    // wave waits for another.  Longer rows do not fit in LDS.  Both take k in the same order: the same bits.
    if (fmt != QMM_Q4_K || shared_fmt != QMM_Q4_K || K > 512)
        return launch_moe_gemm_fmt(fmt, shared_fmt, W, Wsh, ebytes, tiles, counts, max_tiles, rowtab, A, D, N, K,
                                   (hipStream_t)stream);
    // two weight blocks a unit; one where rows of one block and at most four of those leave a tile too few units (1000 x 256,
    // 64 experts, 96 / 512 / 4096 tokens 7.2 / 12.9 / 37.6 against 10.1 / 13.4 / 34.8; 2048 x 256 12.5 / 25.1 / 113 against 11.3 / 23.7 / 96)
    const int nb = (N + XBW - 1) / XBW, bpu = K == 256 && nb <= 4 ? 1 : 2;
    const XArgs a{(const uint8_t*)W, (const uint8_t*)Wsh, ebytes, tiles, counts, rowtab, A, D, N, nb, N, max_tiles, bpu};
    return K == 512 ? launch_moe_gemm_as<2>(a, max_tiles, (hipStream_t)stream) : launch_moe_gemm_as<1>(a, max_tiles, (hipStream_t)stream);
}

int qmm_moe_gemm_gate_up_bf16(int fmt, int shared_fmt, const void* Wg, const void* Wgsh, const void* Wu, const void* Wush,
                              size_t ebytes, const qmm_moe_tile* tiles, const int* counts, int max_tiles, const int* rowtab,
                              const uint16_t* A, uint16_t* H, int N, int K, void* stream) {
    if (fmt != QMM_Q4_K || shared_fmt != QMM_Q4_K) return QMM_ERR_FORMAT;
    if (!Wg || !Wgsh || !Wu || !Wush || !tiles || !counts || !A || !H) return QMM_ERR_NULL;
    if (N <= 0 || K <= 0 || K % 256 != 0 || max_tiles < 0) return QMM_ERR_SHAPE;
    if (max_tiles == 0) return QMM_OK;
    return launch_moe_gate_up_tile(Wg, Wgsh, Wu, Wush, ebytes, tiles, counts, max_tiles, rowtab, A, H, N, K, (hipStream_t)stream);
}

int qmm_moe_silu_bf16(const float* gate, const float* up, uint16_t* h, size_t n, void* stream) {
    if (!gate || !up || !h) return QMM_ERR_NULL;
    if (n == 0) return QMM_OK;
    hipLaunchKernelGGL(k_moe_silu_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, gate, up, h, n);
    QMM_LAUNCH_CHECK();
    return QMM_OK;
}

}  // extern "C"
