"""RMSNorm of few rows: the workgroup-per-row kernel against the one-wave kernel
that a config names, bit for bit (the same sum in the same order, the same
exact division), on both sides of its row limits and of every length's edge."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# [columns]: two, four and eight vectors per lane, each just begun, ragged and full
COLS = [520, 1024, 1032, 2040, 2048, 2056, 3584, 4088, 4096]


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("gamma", [False, True])
def test_few_rows_give_the_one_wave_bits(gpu, cols, gamma):
    from polykernel_amd import kernels as k, runtime as rt

    g = torch.Generator(device=gpu).manual_seed(cols)
    rows_max = 1025
    x = torch.randn(rows_max, cols, generator=g, device=gpu).bfloat16()
    r = torch.randn(rows_max, cols, generator=g, device=gpu).bfloat16()
    x[0, 3] = float("inf")  # rows the fast division cannot take
    x[1] = 0
    r[1] = 0
    x[2] *= 1e30
    x[3] *= 1e-30
    r[3] *= 1e-30
    w = torch.randn(cols, generator=g, device=gpu).bfloat16() if gamma else None
    zero = torch.zeros_like(x)
    for rows in (1, 5, 512, 513, 1024, 1025):
        cfg = rt.default_config("fused_residual_rmsnorm", rows, cols, 0)
        assert cfg["block_m"] == 4 and cfg["vector_width"] == 8
        for res in (r, zero):
            want = k.fused_residual_rmsnorm(x[:rows], res[:rows], w, 1e-6, config=cfg)
            got = k.fused_residual_rmsnorm(x[:rows], res[:rows], w, 1e-6)
            assert torch.equal(_bits(got), _bits(want)), (rows, cols)
        # x + 0 is x (but -0 + 0 = +0: the sign of a zero is not compared)
        got = k.rmsnorm(x[:rows], w, 1e-6)
        finite = torch.isfinite(want)
        assert torch.equal(finite, torch.isfinite(got)), (rows, cols)
        assert torch.equal(got[finite], want[finite]), (rows, cols)
