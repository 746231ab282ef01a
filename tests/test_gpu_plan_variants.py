"""Every variant of the streaming and ring kernels, bf16 and int8, run by name
(the built-in choice depends on fitted constants): each wave refills every slot
of its ring at least twice, the last k-step is ragged, the last row and column
blocks are partial, every epilogue, with the epilogue in place and with K split
over workgroups.  Integer inputs, so every order of the sum is exact."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from polykernel_amd import _lib
from tests.bounds import _int8_exact_inputs
from tests.helpers import bf, from_dev, int_bf16, rng_bf16, to_dev

pytestmark = pytest.mark.gpu

# slice columns x rows of the streams (rings of at most 4 stages, 4 waves that
# take alternate steps of 32 k, int8 of 64), tiles of the rings (at most 4
# stages of 64 k, int8 6)
STREAM = [(n, m) for m in (16, 32, 64) for n in (16, 32, 64, 128)]
RING = [(64, 128), (96, 128), (128, 128), (96, 256), (128, 256), (160, 256)]
INT8_STREAM = [(n, m) for m in (16, 32) for n in (16, 32, 64, 128)]
INT8_RING = [(64, 128), (128, 128), (160, 128), (128, 256), (160, 256)]


def _run(fn, args, tail, M, N, Kd, kernel, bm, bn, splits):
    import torch

    out = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
    ws = torch.full((splits * M * N * 4,), 0xFF, dtype=torch.uint8, device="cuda")
    plan = _lib.Plan(kernel, bm, bn, splits, 0)
    ptr = [None if t is None else t.data_ptr() for t in args]
    _lib.check(getattr(_lib.load(), fn)(tail, ptr[0], ptr[1], *([ptr[2]] if fn == "pk_int8_plan_ex" else []),
                                        out.data_ptr(), *ptr[3 if fn == "pk_int8_plan_ex" else 2:], M, N, Kd,
                                        C.byref(plan), ws.data_ptr(), ws.numel(),
                                        torch.cuda.current_stream().cuda_stream), fn)
    return from_dev(out)


@pytest.mark.parametrize("kernel,bm,bn", [(_lib.PLAN_STREAM, m, n) for n, m in STREAM] +
                         [(_lib.PLAN_RING, m, n) for m, n in RING])
def test_gemm_variant_integer_bit_exact(gpu, oracle, kernel, bm, bn):
    stream = kernel == _lib.PLAN_STREAM
    M, N = (bm - 3, 2 * bn + 8) if stream else (bm + 5, bn + 8)
    for splits, Kd in ((1, 1544), (2, 3112)) if stream else ((1, 808), (2, 1640)):
        print(f"gemm kernel {kernel} {bm}x{bn} splits {splits} K {Kd}", flush=True)
        a, b = int_bf16((M, Kd), 230), int_bf16((Kd, N), 231)
        bias, r = bf(np.random.default_rng(232).integers(-4, 5, size=N)), rng_bf16((M, N), 233)
        da, db, dbias, dr = map(to_dev, (a, b, bias, r))
        for epi, args, want in ((0, (da, db, None, None), oracle.matmul(a, b)),
                                (1, (da, db, dbias, None), oracle.fused_matmul_bias_gelu(a, b, bias)),
                                (2, (da, db, dbias, dr), oracle.fused_matmul_bias_residual(a, b, bias, r)),
                                (3, (da, db, None, dr), oracle.fused_matmul_bias_residual(a, b, None, r))):
            got = _run("pk_gemm_plan_ex", args, epi, M, N, Kd, kernel, bm, bn, splits)
            assert np.array_equal(got, want), (epi, splits)


@pytest.mark.parametrize("kernel,bm,bn", [(_lib.PLAN_STREAM, m, n) for n, m in INT8_STREAM] +
                         [(_lib.PLAN_RING, m, n) for m, n in INT8_RING])
def test_int8_variant_integer_bit_exact(gpu, oracle, kernel, bm, bn):
    stream = kernel == _lib.PLAN_STREAM
    M, N = (bm - 3, 2 * bn + 16) if stream else (bm + 5, bn + 16)
    for splits, Kd in ((1, 3080), (2, 6184)) if stream else ((1, 1192), (2, 2408)):
        print(f"int8 kernel {kernel} {bm}x{bn} splits {splits} K {Kd}", flush=True)
        a, wq, s = _int8_exact_inputs(M, N, Kd, 234)
        r = rng_bf16((M, N), 237)
        da, dw, ds, dr = to_dev(a), to_dev(wq), to_dev(s), to_dev(r)
        plain = oracle.matmul_int8(a, wq, s)
        for epi, want in ((0, plain), (1, oracle.gelu(plain)), (2, oracle.add(plain, r))):
            got = _run("pk_int8_plan_ex", (da, dw, ds, dr), epi, M, N, Kd, kernel, bm, bn, splits)
            assert np.array_equal(got, want), (epi, splits)


def test_plan_that_no_variant_matches_is_refused(gpu):
    a, b = to_dev(int_bf16((64, 72), 238)), to_dev(int_bf16((72, 64), 239))
    for kernel, bm, bn in ((_lib.PLAN_STREAM, 48, 64), (_lib.PLAN_RING, 32, 128), (_lib.PLAN_TILE, 64, 64)):
        with pytest.raises(_lib.PolyKernelError) as ei:
            _run("pk_gemm_plan_ex", (a, b, None, None), 0, 64, 64, 72, kernel, bm, bn, 1)
        assert ei.value.code == _lib.PK_ERR_UNSUPPORTED
