"""The kernels of the prefill GEMMs (gemm_tile.hpp) where their tilings can go wrong: every weight source, sizes
around the edges of each tile (rows 16 .. 256, columns 16 .. 256), K steps that do not divide among the ring's stages, one
row, one column, and every tile of the choice (test_every_tile_is_run asks the library which one a shape takes).

Bound: every product of two bf16 values is exact in f32, so only the K additions round, each by at most 2^-24
of a partial sum, which is at most |a| |w| (Cauchy-Schwarz).  Their errors add up as a random walk: an element is
within 4 sqrt(K) 2^-24 |a| |w| of the float64 product of the same bf16 operands (over six standard deviations of it), and a
matrix within sqrt(K) 2^-24 in the relative 2-norm."""
import numpy as np
import pytest
import torch

from hipster_amd import qmm, synth
from tests.gpu_util import dev

GPU = pytest.mark.gpu
SHAPES = [(1, 70, 512), (70, 1, 512), (17, 33, 1536), (33, 1024, 2560), (40, 6144, 1024), (65, 63, 512), (129, 257, 1024), (300, 2500, 512),
          (193, 8200, 512), (385, 17000, 512), (1100, 300, 1536), (2048, 5120, 512)]
# a shape of every tile, ragged on both sides, two or more rounds of the ring's stages
TILES = [(1, 4099, 1024), (17, 2560, 1536), (2077, 49, 1024), (17, 4147, 1024), (50, 4121, 1536), (100, 5100, 1024), (2311, 775, 512),
         (17, 16439, 512), (67, 17287, 512), (100, 16577, 1536), (259, 13135, 512), (333, 10981, 1024), (294, 16537, 512), (485, 16487, 512), (774, 14659, 512)]
FORMATS = [synth.Q4_K, synth.Q5_K, synth.IQ4_XS, synth.Q6_K_SOA, synth.Q8_0_SOA, synth.Q5_1_SOA]
BF16 = -1


def operands(fmt, M, N, K, seed):
    A = torch.from_numpy(synth.normal_f32(seed, (M, K))).cuda().bfloat16()
    W = dev(synth.matrix(seed + 1, fmt, N, K))
    Wb = torch.zeros((N, K), dtype=torch.int16, device="cuda")
    qmm.dequant_bf16(fmt, W, Wb, N, K)
    Wb = Wb.view(torch.bfloat16)
    return A, W, Wb, A.double() @ Wb.double().t()


def err(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


def check(D, A, Wb, ref, K):
    """every element within its bound, and written"""
    bound = 4 * K ** 0.5 * 2.0 ** -24 * A.double().norm(dim=1)[:, None] * Wb.double().norm(dim=1)[None, :]
    assert ((D.double() - ref).abs() <= bound).all()
    assert err(D, ref) <= K ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("M,N,K", SHAPES + TILES)
@GPU
def test_gemm_wq_tiles(gpu, fmt, M, N, K):
    A, W, Wb, ref = operands(fmt, M, N, K, 7000 + M + N)
    D = torch.full((M, N), float("nan"), device="cuda")
    qmm.gemm_wq(fmt, W, A, D, M, N, K)
    check(D, A, Wb, ref, K)
    # the bf16 GEMM on the dequantised rows is the same chain, rounded once more
    Db = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    qmm.gemm_bf16(A, Wb, Db, M, N, K)
    assert torch.equal(Db.view(torch.int16), D.bfloat16().view(torch.int16))


@pytest.mark.parametrize("fmt", FORMATS + [BF16])
def test_every_tile_is_run(fmt):
    assert sorted({qmm.gemm_tile(fmt, *s) for s in SHAPES + TILES}) == list(range(15))


@pytest.mark.parametrize("fmt,N,K", [(f, n, k) for f in FORMATS for n, k in ((700, 1536), (16500, 512))] +
                         [(synth.Q8_0_SOA, 260, 640), (synth.Q5_1_SOA, 260, 384)])
@GPU
def test_bits_do_not_depend_on_rows_or_columns_of_the_call(gpu, fmt, N, K):
    """the rows of a prompt in chunks of any size, and the columns of a matrix apart or joined: the bits of one call"""
    M = 1600
    A, W, Wb, _ = operands(fmt, M, N, K, 7600 + N)
    full = torch.full((M, N), float("nan"), device="cuda")
    qmm.gemm_wq(fmt, W, A, full, M, N, K)
    tiles = {qmm.gemm_tile(fmt, M, N, K)}
    m0 = 0
    for m in (1, 16, 17, 40, 64, 100, 129, 200, 300, 733):
        D = torch.full((m, N), float("nan"), device="cuda")
        qmm.gemm_wq(fmt, W, A[m0:m0 + m], D, m, N, K)
        assert torch.equal(D.view(torch.int32), full[m0:m0 + m].view(torch.int32)), (m, qmm.gemm_tile(fmt, m, N, K))
        tiles.add(qmm.gemm_tile(fmt, m, N, K))
        m0 += m
    assert m0 == M and len(tiles) >= 3, tiles
    for n0, n in ((0, 3), (3, 100), (103, N - 103)):
        for m in (16, 300):
            D = torch.full((m, n), float("nan"), device="cuda")
            qmm.gemm_wq(fmt, W[n0:n0 + n], A[:m], D, m, n, K)
            assert torch.equal(D.view(torch.int32), full[:m, n0:n0 + n].contiguous().view(torch.int32)), (n, m)


@pytest.mark.parametrize("fmt,K", [(synth.Q8_0_SOA, 128), (synth.Q5_1_SOA, 640), (synth.Q4_K, 256), (synth.Q6_K_SOA, 512)])
@GPU
def test_gemm_wq_short_k(gpu, fmt, K):
    """fewer K steps than the ring has stages, and a last round that is not full"""
    A, W, Wb, ref = operands(fmt, 21, 70, K, 7100 + K)
    D = torch.full((21, 70), float("nan"), device="cuda")
    qmm.gemm_wq(fmt, W, A, D, 21, 70, K)
    assert err(D, ref) <= K ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("fmt,K", [(synth.Q8_0_SOA, 128), (synth.Q8_0_SOA, 640), (synth.Q5_1_SOA, 128), (synth.Q5_1_SOA, 896)])
@GPU
def test_bytes_behind_the_matrix_do_not_matter(gpu, fmt, K):
    """a last chunk of scales that is not full, of the last row: what lies behind the matrix (scales of NaN here) is not
    read into any result, in a tile by waves of 32 rows and in one by producers"""
    for M, N in ((300, 4097), (5, 37)):
        W = synth.matrix(7210 + K, fmt, N, K)
        buf = torch.full((W.size + 256,), 255, dtype=torch.uint8, device="cuda")
        buf[:W.size] = dev(W).reshape(-1)
        A = torch.from_numpy(synth.normal_f32(7211, (M, K))).cuda().bfloat16()
        D, E = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
        qmm.gemm_wq(fmt, buf[:W.size], A, D, M, N, K)
        buf[W.size:] = 0
        qmm.gemm_wq(fmt, buf[:W.size], A, E, M, N, K)
        assert torch.isfinite(D).all() and torch.equal(D, E)


@GPU
def test_gemm_bf16_odd_step_count_and_strides(gpu):
    """K = 192 (three steps) and operands that are views of wider matrices, garbage (NaN) around them"""
    M, N, K = 45, 300, 192
    A = torch.full((M, 256), float("nan"), device="cuda", dtype=torch.bfloat16)
    W = torch.full((N, 200), float("nan"), device="cuda", dtype=torch.bfloat16)
    A[:, :K] = torch.from_numpy(synth.normal_f32(7200, (M, K))).cuda().bfloat16()
    W[:, :K] = torch.from_numpy(synth.normal_f32(7201, (N, K))).cuda().bfloat16()
    D = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    qmm.gemm_bf16_ld(A, 256, W, 200, D, M, N, K)
    a, w = A[:, :K].double(), W[:, :K].double()
    ref = a @ w.t()
    # the sum's bound, then one rounding to 8 bits
    assert ((D.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 4 * K ** 0.5 * 2.0 ** -24 * a.norm(dim=1)[:, None] * w.norm(dim=1)[None, :]).all()


@GPU
def test_gemm_bf16_rows_too_far_apart_for_any_tile(gpu):
    """row strides of 160 and 155 million elements, of A and of W: 16 rows of either exceed a buffer resource, so the call runs in
    parts; the bits of the same rows side by side"""
    M, N, K = 20, 27, 192
    lda, ldw = 160_000_000, 155_000_000
    a = torch.from_numpy(synth.normal_f32(7220, (M, K))).cuda().bfloat16()
    w = torch.from_numpy(synth.normal_f32(7221, (N, K))).cuda().bfloat16()
    want, D = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    qmm.gemm_bf16(a, w, want, M, N, K)
    buf = torch.empty(max((M - 1) * lda, (N - 1) * ldw) + K, dtype=torch.bfloat16, device="cuda")
    A = buf.as_strided((M, K), (lda, 1))
    A.copy_(a)
    qmm.gemm_bf16_ld(A, lda, w, K, D, M, N, K)
    assert torch.equal(D.view(torch.int16), want.view(torch.int16))
    D.fill_(float("nan"))
    W = buf.as_strided((N, K), (ldw, 1))
    W.copy_(w)
    qmm.gemm_bf16_ld(a, K, W, ldw, D, M, N, K)
    assert torch.isfinite(D.float()).all() and torch.equal(D.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(40, 96, 768), (300, 4200, 256)])
@GPU
def test_gemm_wq_rows_do_not_mix(gpu, M, N, K):
    """an infinite activation spoils its own row only, also beside rows and K steps that a tile pads"""
    A, W, Wb, ref = operands(synth.Q4_K, M, N, K, 7300)
    A[7, 5] = float("inf")
    D = torch.zeros((M, N), device="cuda")
    qmm.gemm_wq(synth.Q4_K, W, A, D, M, N, K)
    keep = np.arange(M) != 7
    assert not torch.isfinite(D[7]).any()
    assert err(D[keep], ref[torch.from_numpy(keep)]) <= K ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("fmt,N,K", [(synth.Q4_K, 130, 256), (synth.Q4_K, 70, 768), (synth.Q5_K, 128, 512), (synth.IQ4_XS, 33, 768), (synth.Q8_0_SOA, 257, 192),
                                     (synth.Q5_1_SOA, 2560, 640), (synth.Q5_1_SOA, 100, 96), (synth.Q8_0_SOA, 40, 64)])
@pytest.mark.parametrize("gather", [True, False])
@GPU
def test_grouped_tiles(gpu, fmt, N, K, gather):
    """every number of row blocks (tiles of 1, 31, 32, 33, 64, 65, 97, 128 rows), partial column blocks, K of a
    partial chunk of steps (Q8_0 K = 64 and 192) and Q5_1 rows that steps of 64 do not divide, routed and shared tiles"""
    sizes = [1, 31, 32, 33, 64, 65, 97, 128]
    E, rows = len(sizes) - 1, sum(sizes)
    sf = synth.Q8_0_SOA if fmt != synth.Q8_0_SOA and K % 64 == 0 else fmt
    W, S = dev(synth.experts(7400 + K, fmt, E, N, K)), dev(synth.matrix(7401 + K, sf, N, K))
    deq = lambda f, w: (lambda o: (qmm.dequant_bf16(f, w, o, N, K), o.view(torch.bfloat16).double())[1])(   # noqa: E731
        torch.zeros((N, K), dtype=torch.int16, device="cuda"))
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    tiles = np.array([[e, starts[e], sizes[e]] for e in range(E)] + [[-1, starts[E], sizes[E]]], np.int32)
    A = torch.from_numpy(synth.normal_f32(7402, (rows if not gather else 200, K))).cuda().bfloat16()
    rt = synth.rng(7403).integers(0, A.shape[0], rows).astype(np.int32) if gather else None
    D = torch.full((rows, N), float("nan"), device="cuda")
    qmm.moe_gemm_bf16(fmt, sf, W, S, W[0].numel(), dev(tiles), dev(np.array([E, 1], np.int32)), E + 1,
                      dev(rt) if gather else None, A, D, N, K)
    idx = torch.from_numpy(rt.astype(np.int64)).cuda() if gather else torch.arange(rows, device="cuda")
    for e, (k0, n) in enumerate(zip(starts, sizes)):
        ref = A[idx[k0:k0 + n]].double() @ (deq(fmt, W[e]) if e < E else deq(sf, S)).t()
        assert err(D[k0:k0 + n], ref) <= K ** 0.5 * 2.0 ** -24, (e, n)


@pytest.mark.parametrize("N,K", [(64, 256), (70, 768), (1, 512), (130, 2048)])
@GPU
def test_gate_up_tiles(gpu, N, K):
    """the fused gate/up call at every number of row blocks and partial blocks of 64 rows: bit for bit the two
    grouped GEMMs and silu * up it stands for"""
    sizes = [1, 31, 32, 33, 64, 65, 97, 128]
    E, rows = len(sizes) - 1, sum(sizes)
    W = [dev(synth.experts(7500 + i, synth.Q4_K, E, N, K)) for i in range(2)]
    S = [dev(synth.matrix(7502 + i, synth.Q4_K, N, K)) for i in range(2)]
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    tiles = dev(np.array([[e, starts[e], sizes[e]] for e in range(E)] + [[-1, starts[E], sizes[E]]], np.int32))
    counts = dev(np.array([E, 1], np.int32))
    # weights of these blocks are of order 1e3: the activations keep gate and up in silu's range
    A = (torch.from_numpy(synth.normal_f32(7504, (200, K))).cuda() * 1e-4).bfloat16()
    rt = dev(synth.rng(7505).integers(0, 200, rows).astype(np.int32))
    h, h2 = (torch.zeros((rows, N), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    eb = W[0][0].numel()
    qmm.moe_gemm_gate_up_bf16(synth.Q4_K, synth.Q4_K, W[0], S[0], W[1], S[1], eb, tiles, counts, E + 1, rt, A, h, N, K)
    gu = [torch.full((rows, N), float("nan"), device="cuda") for _ in range(2)]
    for i in range(2):
        qmm.moe_gemm_bf16(synth.Q4_K, synth.Q4_K, W[i], S[i], eb, tiles, counts, E + 1, rt, A, gu[i], N, K)
    qmm.moe_silu_bf16(gu[0], gu[1], h2, rows * N)
    assert torch.isfinite(h.float()).all() and h.float().abs().max() > 0
    assert torch.equal(h.view(torch.int16), h2.view(torch.int16))


@pytest.mark.parametrize("fmt,K", [(synth.Q4_K, 256), (synth.Q4_K, 512), (synth.Q4_K, 768), (synth.Q5_K, 512), (synth.Q5_1_SOA, 640)])
@GPU
def test_grouped_rows_beyond_a_buffer_offset(gpu, fmt, K):
    """an A of more than 4 GiB, past the span of the gather's 32-bit offsets: tiles of near, of far and of both kinds of rows give the
    bits that the same rows give in a small A, gathered (the fused gate/up call too) and in sorted order"""
    N, rows_a = 130, 2 ** 32 // (2 * K) + 4000
    near, far = torch.arange(0, 200), torch.arange(rows_a - 300, rows_a)
    sizes = [128, 64, 97, 128, 5]
    g = synth.rng(7800)
    pick = [near[:128], far[:64], torch.cat([near, far])[torch.from_numpy(g.permutation(500)[:97])],
            torch.cat([near, far])[torch.from_numpy(g.permutation(500)[:128])], far[-5:]]
    rt = torch.cat(pick).int().cuda()
    E, starts = len(sizes) - 1, np.concatenate([[0], np.cumsum(sizes)[:-1]])
    tiles = dev(np.array([[e, starts[e], sizes[e]] for e in range(E)] + [[-1, starts[E], sizes[E]]], np.int32))
    counts = dev(np.array([E, 1], np.int32))
    W, S = dev(synth.experts(7801, fmt, E, N, K)), dev(synth.matrix(7802, fmt, N, K))
    A = torch.empty((rows_a, K), dtype=torch.bfloat16, device="cuda")
    for r in (near, far):
        A[r.cuda()] = (torch.from_numpy(synth.normal_f32(7803 + int(r[0]) % 7, (len(r), K))).cuda() * 1e-3).bfloat16()
    small = A[rt.long()].contiguous()
    n, eb = len(rt), W[0].numel()
    D, D2 = (torch.full((n, N), float("nan"), device="cuda") for _ in range(2))
    qmm.moe_gemm_bf16(fmt, fmt, W, S, eb, tiles, counts, E + 1, rt, A, D, N, K)
    qmm.moe_gemm_bf16(fmt, fmt, W, S, eb, tiles, counts, E + 1, None, small, D2, N, K)
    assert torch.isfinite(D2).all() and torch.equal(D.view(torch.int32), D2.view(torch.int32))
    if fmt == synth.Q4_K:
        H, H2 = (torch.full((n, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        qmm.moe_gemm_gate_up_bf16(fmt, fmt, W, S, W, S, eb, tiles, counts, E + 1, rt, A, H, N, K)
        qmm.moe_gemm_gate_up_bf16(fmt, fmt, W, S, W, S, eb, tiles, counts, E + 1, None, small, H2, N, K)
        assert torch.isfinite(H2.float()).all() and torch.equal(H.view(torch.int16), H2.view(torch.int16))
    # sorted order: consecutive rows of A, the last of them far
    k0 = rows_a - 300
    one = dev(np.array([[0, k0, 128], [1, k0 + 128, 100]], np.int32))
    big = torch.full((rows_a, 2), float("nan"), device="cuda")
    qmm.moe_gemm_bf16(fmt, fmt, W[:, :2].contiguous(), S[:2].contiguous(), 2 * W[0, 0].numel(), one, dev(np.array([2, 0], np.int32)), 2, None, A, big, 2, K)
    near2 = dev(np.array([[0, 0, 128], [1, 128, 100]], np.int32))
    few = torch.full((228, 2), float("nan"), device="cuda")
    qmm.moe_gemm_bf16(fmt, fmt, W[:, :2].contiguous(), S[:2].contiguous(), 2 * W[0, 0].numel(), near2, dev(np.array([2, 0], np.int32)), 2, None,
                      A[k0:k0 + 228].contiguous(), few, 2, K)
    assert torch.isfinite(few).all() and torch.equal(big[k0:k0 + 228].view(torch.int32), few.view(torch.int32))
