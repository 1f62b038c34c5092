"""The tile kernel of the prefill GEMMs (gemm_tile.hpp) where its tilings can go wrong: every weight
source, sizes around the edges of each tile (rows 32, 64, 128, 192; columns 32, 64, 128, 256), K steps that do not
divide among the K groups, one row, one column, and a shape per tile choice.

Bound: every product of two bf16 values is exact in f32, so only the K additions round.  Their errors add
up as a random walk, each at most 2^-24 of a partial sum that grows like sqrt(k): sqrt(K) 2^-24 relative
in the 2-norm, against the float64 product of the same bf16 operands."""
import numpy as np
import pytest
import torch

from hipster_amd import qmm, synth
from tests.gpu_util import dev

pytestmark = pytest.mark.gpu
SHAPES = [(1, 70, 512), (70, 1, 512), (17, 33, 1536), (33, 1024, 2560), (40, 6144, 1024), (65, 63, 512), (129, 257, 1024), (300, 2500, 512),
          (193, 8200, 512), (385, 17000, 512), (1100, 300, 1536), (2048, 5120, 512)]


def operands(fmt, M, N, K, seed):
    A = torch.from_numpy(synth.normal_f32(seed, (M, K))).cuda().bfloat16()
    W = dev(synth.matrix(seed + 1, fmt, N, K))
    Wb = torch.zeros((N, K), dtype=torch.int16, device="cuda")
    qmm.dequant_bf16(fmt, W, Wb, N, K)
    Wb = Wb.view(torch.bfloat16)
    return A, W, Wb, A.double() @ Wb.double().t()


def err(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("fmt", [synth.Q4_K, synth.Q5_K, synth.IQ4_XS, synth.Q6_K_SOA, synth.Q8_0_SOA, synth.Q5_1_SOA])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_wq_tiles(gpu, fmt, M, N, K):
    A, W, Wb, ref = operands(fmt, M, N, K, 7000 + M + N)
    D = torch.full((M, N), float("nan"), device="cuda")
    qmm.gemm_wq(fmt, W, A, D, M, N, K)
    assert err(D, ref) <= K ** 0.5 * 2.0 ** -24
    # the bf16 GEMM takes the same tile and K order, but lanes of some formats hold k in another order: the same
    # sums within the bound, then one rounding to bf16 (8 bits: 2^-8 at most)
    Db = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
    qmm.gemm_bf16(A, Wb, Db, M, N, K)
    assert err(Db, ref) <= 2.0 ** -8


@pytest.mark.parametrize("fmt,K", [(synth.Q8_0_SOA, 128), (synth.Q5_1_SOA, 640), (synth.Q4_K, 256), (synth.Q6_K_SOA, 512)])
def test_gemm_wq_short_k(gpu, fmt, K):
    """fewer K steps than K groups, and a last group without a step"""
    A, W, Wb, ref = operands(fmt, 21, 70, K, 7100 + K)
    D = torch.full((21, 70), float("nan"), device="cuda")
    qmm.gemm_wq(fmt, W, A, D, 21, 70, K)
    assert err(D, ref) <= K ** 0.5 * 2.0 ** -24


def test_gemm_bf16_odd_step_count_and_strides(gpu):
    """K = 192 (three steps) and operands that are views of wider matrices, garbage (NaN) around them"""
    M, N, K = 45, 300, 192
    A = torch.full((M, 256), float("nan"), device="cuda", dtype=torch.bfloat16)
    W = torch.full((N, 200), float("nan"), device="cuda", dtype=torch.bfloat16)
    A[:, :K] = torch.from_numpy(synth.normal_f32(7200, (M, K))).cuda().bfloat16()
    W[:, :K] = torch.from_numpy(synth.normal_f32(7201, (N, K))).cuda().bfloat16()
    D = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
    qmm.gemm_bf16_ld(A, 256, W, 200, D, M, N, K)
    assert err(D, A[:, :K].double() @ W[:, :K].double().t()) <= 2.0 ** -8


def test_gemm_wq_rows_do_not_mix(gpu):
    """an infinite activation spoils its own row only, also beside rows and K steps that a tile pads"""
    M, N, K = 40, 96, 768
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
