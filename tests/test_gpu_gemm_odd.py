"""Products of at most 64 rows whose weight rows start at any element (N % 8 != 0
or an unaligned B): every slice width and row block, ragged last chunks and
k-steps, against the oracle; integer inputs, so every order of the sum is
exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.helpers import from_dev, int_bf16, rng_bf16, to_dev

pytestmark = pytest.mark.gpu


# N within one chunk, one over a slice of 32, 64 and 128 columns, and on both
# sides of the width limits (8192, 20480); K of one chunk, below, at and past a
# k-step of 32 and past a round of the ring of every wave (8 waves x 5 steps)
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,Kd", [(9, 8), (15, 40), (33, 32), (262, 520), (1029, 1352), (8191, 264), (8193, 1064),
                                  (20479, 72), (20481, 424)])
def test_odd_rows_integer_bit_exact(gpu, oracle, M, N, Kd):
    from polykernel_amd import kernels

    print(f"odd {M}x{N}x{Kd}", flush=True)
    a, b = int_bf16((M, Kd), 214), int_bf16((Kd, N), 215)
    assert np.array_equal(from_dev(kernels.matmul(to_dev(a), to_dev(b))), oracle.matmul(a, b))


@pytest.mark.parametrize("off", [1, 2, 7])
@pytest.mark.parametrize("M,N,Kd", [(5, 64, 40), (20, 8200, 64), (40, 20488, 40)])
def test_unaligned_weights_and_infinities(gpu, oracle, M, N, Kd, off):
    """B at any element, whose neighbours in memory and last row hold infinities."""
    from polykernel_amd import kernels

    a, b = int_bf16((M, Kd), 216), int_bf16((Kd, N), 217)
    b[Kd - 1, ::3] = 0x7F80
    a[:, Kd - 1] = 0x3F80
    buf = torch.full((Kd * N + 16,), float("inf"), dtype=torch.bfloat16, device="cuda")
    buf[off:off + Kd * N] = to_dev(b).reshape(-1)
    got = from_dev(kernels.matmul(to_dev(a), buf[off:off + Kd * N].view(Kd, N)))
    assert np.array_equal(got, oracle.matmul(a, b))


@pytest.mark.parametrize("M,N,Kd", [(1, 2049, 896), (33, 8195, 2048)])
def test_odd_rmsnorm_matmul_is_its_composition(gpu, M, N, Kd):
    from polykernel_amd import kernels

    x, g, w = (to_dev(rng_bf16(s, 218 + i)) for i, s in enumerate([(M, Kd), (Kd,), (Kd, N)]))
    got = kernels.fused_rmsnorm_matmul(x, w, g, 1e-6)
    want = kernels.matmul(kernels.rmsnorm(x, g, 1e-6), w)
    assert torch.equal(got, want)
