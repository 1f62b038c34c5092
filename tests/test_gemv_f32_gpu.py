"""The f32-activation Q4_K GEMV on the f32 matrix cores: every column of every launch split is bit for bit the
one-column VALU kernel's (both are the same chain of fused multiply-adds), over row counts that leave partial row
groups, idle waves and a second walk over the rows, and every number of pair iterations (K 256 .. 6144)."""
import pytest
import torch

from hipster_amd import qmm, synth
from tests.gpu_util import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 256), (5, 768), (1022, 1280), (1023, 2304), (70, 3328), (2049, 4352), (9001, 5120), (333, 6144)])
def test_columns_are_bitwise_the_one_column_kernel(gpu, N, K):
    W = dev(synth.matrix(7500 + K, synth.Q4_K, N, K))
    x = dev(synth.normal_f32(7501 + N, (8, K)))
    one = torch.full((8, N), float("nan"), device="cuda")
    for c in range(8):
        qmm.gemv_q4_K_f32(W, x[c:c + 1].contiguous(), one[c:c + 1], N, K, 1)
    for ncol in (3, 4, 5, 7, 8):
        y = torch.full((ncol, N), float("nan"), device="cuda")
        qmm.gemv_q4_K_f32(W, x[:ncol].contiguous(), y, N, K, ncol)
        assert torch.equal(y, one[:ncol]), ncol


def test_infinite_column_stays_in_its_column(gpu):
    N, K = 40, 512
    W = dev(synth.matrix(7600, synth.Q4_K, N, K))
    x = dev(synth.normal_f32(7601, (4, K)))
    ref = torch.zeros((4, N), device="cuda")
    qmm.gemv_q4_K_f32(W, x, ref, N, K, 4)
    x[2, 7] = float("inf")
    y = torch.zeros((4, N), device="cuda")
    qmm.gemv_q4_K_f32(W, x, y, N, K, 4)
    assert torch.equal(y[[0, 1, 3]], ref[[0, 1, 3]])
    assert not torch.isfinite(y[2]).any()
