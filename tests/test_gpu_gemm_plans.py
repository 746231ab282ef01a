"""GEMMs of decode and prompt size through the entry points' own choice of
kernel, at ragged edges, with every epilogue, with and without K splits.  (Each
variant of the streaming and ring kernels by name, over several rounds of its
ring: test_gpu_plan_variants.py.)"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from polykernel_amd import synth
from tests.bounds import _gate_bad, _int8_exact_inputs
from tests.helpers import bf, from_dev, int_bf16, rng_bf16, to_dev

pytestmark = pytest.mark.gpu


# rows at the edges of the 16-row blocks; K a multiple of 32 or only of 8 (40,
# 520: a last step with 8 rows); N within one slice, ragged, and with whole
# slices of 128, 64, 32 and 16 columns (50256, 16384, 8192, 3072)
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,Kd", [(8, 8), (8, 40), (264, 512), (1000, 520), (3072, 768), (8192, 1032),
                                  (16384, 256), (50256, 40)])
def test_small_m_gemm_integer_bit_exact(gpu, oracle, M, N, Kd):
    _check_integer(oracle, M, N, Kd)


# above 64 rows: one row over a tile of 64 to 160 rows, K below, at and above a
# k-tile of 64 with tails of 8 to 56 (the tile kernels for a short K, the ring
# kernel for a long one)
@pytest.mark.parametrize("M,N,Kd", [(65, 8, 8), (97, 136, 72), (129, 264, 520), (272, 6592, 40), (391, 6680, 64),
                                    (514, 6744, 120), (879, 6456, 72), (1060, 7184, 200), (161, 2056, 1336)])
def test_ring_gemm_integer_bit_exact(gpu, oracle, M, N, Kd):
    _check_integer(oracle, M, N, Kd)


def _check_integer(oracle, M, N, Kd):
    from polykernel_amd import kernels

    print(f"gemm {M}x{N}x{Kd}", flush=True)
    a, b = int_bf16((M, Kd), 114), int_bf16((Kd, N), 115)
    bias, r = bf(np.random.default_rng(116).integers(-4, 5, size=N)), rng_bf16((M, N), 117)
    da, db, dbias, dr = map(to_dev, (a, b, bias, r))
    assert np.array_equal(from_dev(kernels.matmul(da, db)), oracle.matmul(a, b))
    assert np.array_equal(from_dev(kernels.fused_matmul_bias_gelu(da, db, dbias)),
                          oracle.fused_matmul_bias_gelu(a, b, bias))
    for bb, dbb in ((bias, dbias), (None, None)):
        assert np.array_equal(from_dev(kernels.fused_matmul_bias_residual(da, db, dbb, dr)),
                              oracle.fused_matmul_bias_residual(a, b, bb, r))


@pytest.mark.parametrize("M,N,Kd", [(5, 72, 40), (70, 72, 40), (70, 72, 200)])
def test_gemm_rows_past_k_do_not_leak(gpu, oracle, M, N, Kd):
    """The last k-step of a ragged K reaches past it; the memory a clamped load
    repeats there holds infinities, which must not reach a sum."""
    from polykernel_amd import kernels

    a, b = int_bf16((M, Kd), 118), int_bf16((Kd, N), 119)
    b[Kd - 1] = 0x7F80  # +inf weights in the last valid row, against zero and nonzero activations
    a[:, Kd - 1] = 0x3F80
    a[2, Kd - 1] = 0  # 0 * inf = NaN
    got, want = from_dev(kernels.matmul(to_dev(a), to_dev(b))), oracle.matmul(a, b)
    rest = np.arange(M) != 2
    assert np.array_equal(got[rest], want[rest])
    assert np.all((got[2] & 0x7F80) == 0x7F80) and np.all(got[2] & 0x7F)


# (M, d, F): K splits in both products, in one of them, ragged widths and K
@pytest.mark.parametrize("M,d,F", [(1, 512, 2048), (16, 1024, 4096), (17, 768, 3072), (33, 520, 2056),
                                   (64, 2048, 1000), (5, 4096, 512), (64, 4096, 4096), (65, 512, 2048),
                                   (100, 768, 3072), (333, 520, 2056), (501, 1024, 4096), (777, 2048, 4096)])
def test_mlp_block_stages(gpu, M, d, F):
    """launch_mlp_block's two GEMMs, each held to the fp32 error model on the
    operands it read (from the workspace), with the whole workspace and with
    only the rows (no room for split partials)."""
    import torch

    from polykernel_amd import _lib, kernels

    lib = _lib.load()
    x = to_dev(synth.normal_bf16((M, d), 140))
    g = to_dev(synth.normal_bf16((d,), 141, 0.1, 1.0))
    w1, w2 = (to_dev(synth.normal_bf16(s, 142 + i, 1 / np.sqrt(s[0]))) for i, s in enumerate(((d, F), (F, d))))
    b1, b2 = to_dev(synth.normal_bf16((F,), 144, 0.02)), to_dev(synth.normal_bf16((d,), 145, 0.02))
    up = lambda v: (v + 255) & ~255  # noqa: E731
    rows = up(2 * M * d) + up(2 * M * F)
    assert lib.pk_mlp_block_workspace_size(M, d, F) >= rows
    for size in (lib.pk_mlp_block_workspace_size(M, d, F), rows):
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")
        out = torch.empty_like(x)
        _lib.check(lib.launch_mlp_block(x.data_ptr(), g.data_ptr(), w1.data_ptr(), b1.data_ptr(), w2.data_ptr(),
                                        b2.data_ptr(), out.data_ptr(), M, d, F, ctypes.c_float(1e-6), ws.data_ptr(),
                                        size, torch.cuda.current_stream().cuda_stream), "launch_mlp_block")
        a = ws[:2 * M * d].view(torch.bfloat16).view(M, d)
        h = ws[up(2 * M * d):up(2 * M * d) + 2 * M * F].view(torch.bfloat16).view(M, F)
        assert torch.equal(a, kernels.rmsnorm(x, g, 1e-6))
        assert _gate_bad(1, a.contiguous(), w1, h.contiguous(), bias=b1) == 0, (M, d, F, size)
        assert _gate_bad(2, h.contiguous(), w2, out, bias=b2, r=x) == 0, (M, d, F, size)
    assert lib.launch_mlp_block(x.data_ptr(), g.data_ptr(), w1.data_ptr(), b1.data_ptr(), w2.data_ptr(),
                                b2.data_ptr(), out.data_ptr(), M, d, F, ctypes.c_float(1e-6), ws.data_ptr(),
                                rows - 1, None) == _lib.PK_ERR_WORKSPACE


@pytest.mark.parametrize("M,N,Kd", [(16, 768, 3072), (33, 2048, 4096), (7, 512, 1032), (130, 768, 3072)])
def test_rmsnorm_matmul_split(gpu, M, N, Kd):
    """RMSNorm -> MatMul with the split partials behind the normalised rows in
    the library workspace, eager and captured (the replay keeps the eager bits)."""
    import torch

    from polykernel_amd import kernels

    x = to_dev(synth.normal_bf16((M, Kd), 150))
    g = to_dev(synth.normal_bf16((Kd,), 151, 0.1, 1.0))
    w = to_dev(synth.normal_bf16((Kd, N), 152, 1 / np.sqrt(Kd)))
    got = kernels.fused_rmsnorm_matmul(x, w, g, 1e-6)
    assert _gate_bad(0, kernels.rmsnorm(x, g, 1e-6), w, got) == 0
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        kernels.fused_rmsnorm_matmul(x, w, g, 1e-6)
        torch.cuda.synchronize()
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr, stream=s):
            out = kernels.fused_rmsnorm_matmul(x, w, g, 1e-6)
    for _ in range(3):
        out.fill_(0)
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), got.view(torch.int16))
        assert torch.equal(kernels.fused_rmsnorm_matmul(x, w, g, 1e-6).view(torch.int16), got.view(torch.int16))


# the int8 K-split stream: slices of 16 to 128 columns (few, ragged, whole), rows
# at the edges of its 16- and 32-row blocks, K tails of 8 to 56, K splits in
# library scratch (long K) -- and above 32 rows K tails, K splits (512 columns,
# long K), N with a ragged 16-column chunk
@pytest.mark.parametrize("M,N,Kd", [(1, 16, 8), (16, 16, 72), (17, 144, 520), (5, 1040, 520), (32, 3968, 1472),
                                    (3, 1472, 3968), (16, 2048, 8200), (32, 4096, 4160), (16, 16384, 136),
                                    (9, 11008, 1024), (20, 16384, 512), (33, 16, 8), (65, 144, 72), (129, 272, 520), (48, 512, 4096), (300, 2064, 1032),
                                    (391, 6688, 64), (300, 12288, 64), (879, 6464, 72), (1060, 7184, 136),
                                    (600, 1040, 4104)])
def test_int8_plans_integer_bit_exact(gpu, oracle, M, N, Kd):
    from polykernel_amd import _lib, kernels

    print(f"int8 {M}x{N}x{Kd}", flush=True)
    a, wq, s = _int8_exact_inputs(M, N, Kd, 160)
    r = rng_bf16((M, N), 163)
    da, dw, ds, dr = to_dev(a), to_dev(wq), to_dev(s), to_dev(r)
    plain = oracle.matmul_int8(a, wq, s)
    got = kernels.matmul_int8(da, dw, ds)
    assert np.array_equal(from_dev(got), plain)
    assert np.array_equal(from_dev(kernels.matmul_int8_ex(1, da, dw, ds)), oracle.gelu(plain))
    assert np.array_equal(from_dev(kernels.matmul_int8_ex(2, da, dw, ds, dr)), oracle.add(plain, r))
    import torch

    out = torch.empty_like(got)
    rc = _lib.load().launch_matmul_int8_noalloc(da.data_ptr(), dw.data_ptr(), ds.data_ptr(), out.data_ptr(), M, N, Kd,
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.PK_ERR_WORKSPACE or (rc == 0 and torch.equal(out.view(torch.int16), got.view(torch.int16)))
