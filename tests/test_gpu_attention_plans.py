"""Attention of 1 to 4 queries per head (attention_decode_kernel): batch and
wave edges of the key range, key splits, causal limits, the fused append; and
the flash kernel's built-in choices at head dim 64 and at any cache length."""
from __future__ import annotations

import numpy as np
import pytest

from polykernel_amd import metrics as mt
from polykernel_amd import synth
from tests.bounds import _att_bound_bad
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _check(oracle, got, q, k, v, causal):
    want = oracle.attention_prefill(q, k, v, None, causal)
    rep = mt.report(got, want)
    assert rep.cosine >= 0.999 and rep.pcc >= 0.99, rep
    assert _att_bound_bad(oracle, got, want, q, k, v, causal) == 0, rep


# keys: one, below / at / above a batch (32 keys at D 128, 64 at 64), the 8
# waves' batches, and enough for several key splits; heads that split and not
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (2, 3, 1, 31), (1, 2, 1, 64), (1, 2, 2, 65), (2, 2, 3, 255),
                                        (1, 3, 4, 257), (1, 2, 1, 4099), (1, 2, 4, 2050), (9, 29, 1, 70)])
@pytest.mark.parametrize("causal", [True, False])
def test_decode_attention(gpu, oracle, B, H, Sq, Skv, D, causal):
    from polykernel_amd import kernels

    print(f"decode attention B{B} H{H} Sq{Sq} Skv{Skv} D{D} causal={causal}", flush=True)
    q = synth.normal_bf16((B, H, Sq, D), 180)
    k = synth.normal_bf16((B, H, Skv, D), 181)
    v = synth.normal_bf16((B, H, Skv, D), 182)
    got = from_dev(kernels.attention_prefill(to_dev(q), to_dev(k), to_dev(v), None, causal))
    _check(oracle, got, q, k, v, causal)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Sc,spare", [(1, 2, 1, 0, 0), (2, 2, 1, 127, 5), (1, 3, 3, 128, 0), (2, 2, 4, 1021, 2),
                                             (1, 2, 2, 2047, 0)])
def test_decode_append_attention(gpu, oracle, B, H, Sq, Sc, spare, D):
    """The appended rows land in the caches bit for bit, nothing else moves, and
    the new rows are seen although the cache is written by the same launch."""
    from polykernel_amd import kernels

    print(f"decode append B{B} H{H} Sq{Sq} Sc{Sc} D{D}", flush=True)
    q, kn, vn = (synth.normal_bf16((B, H, Sq, D), 183 + i) for i in range(3))
    kc, vc = (synth.normal_bf16((B, H, Sc + Sq + spare, D), 186 + i) for i in range(2))
    dk, dv = to_dev(kc), to_dev(vc)
    got = from_dev(kernels.fused_kv_append_attention(to_dev(q), to_dev(kn), to_dev(vn), dk, dv, Sc))
    for cache, new, dev in ((kc, kn, dk), (vc, vn, dv)):
        cache[:, :, Sc:Sc + Sq] = new
        assert np.array_equal(from_dev(dev), cache)
    _check(oracle, got, q, kc[:, :, :Sc + Sq], vc[:, :, :Sc + Sq], True)


# more than 4 queries: the step that holds row S_cache reads cached and new
# more than 4 queries behind a cache of any length: the append is a launch of its
# own unless the cache ends on a key step of the tile; with key splits (few heads)
# and with D 64 in one round (half ring) and several (pairs)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Sc", [(1, 2, 5, 1), (1, 2, 70, 127), (1, 2, 70, 129), (2, 3, 33, 1000), (1, 4, 600, 65),
                                       (1, 2, 333, 1501), (2, 16, 600, 961), (3, 40, 130, 201)])
def test_flash_append_any_cache_length(gpu, oracle, B, H, Sq, Sc, D):
    from polykernel_amd import kernels

    print(f"flash append B{B} H{H} Sq{Sq} Sc{Sc} D{D}", flush=True)
    q, kn, vn = (synth.normal_bf16((B, H, Sq, D), 190 + i) for i in range(3))
    kc, vc = (synth.normal_bf16((B, H, Sc + Sq + 3, D), 193 + i) for i in range(2))
    dk, dv = to_dev(kc), to_dev(vc)
    got = from_dev(kernels.fused_kv_append_attention(to_dev(q), to_dev(kn), to_dev(vn), dk, dv, Sc))
    for cache, new, dev in ((kc, kn, dk), (vc, vn, dv)):
        cache[:, :, Sc:Sc + Sq] = new
        assert np.array_equal(from_dev(dev), cache)
    _check(oracle, got, q, kc[:, :, :Sc + Sq], vc[:, :, :Sc + Sq], True)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("BH,Sq,Skv", [(4, 65, 300), (5, 600, 2500), (300, 70, 200), (130, 200, 700)])
def test_flash_d64_rings(gpu, oracle, BH, Sq, Skv, causal):
    from polykernel_amd import kernels

    q, k, v = (synth.normal_bf16((1, BH, n, 64), 196 + i) for i, n in enumerate((Sq, Skv, Skv)))
    got = from_dev(kernels.attention_prefill(to_dev(q), to_dev(k), to_dev(v), None, causal))
    _check(oracle, got, q, k, v, causal)


# each variant of the built-in choice by name, with key splits of 1, even and odd
# counts, and splits past the last step (25 steps in 8, 10 in 8) or batch (97 and 121
# in 12)
@pytest.mark.parametrize("BH,Sq,Sc,D,append,kernel,block_m,splits,inside", [
    (7, 38, 64, 64, True, "FLASH", 128, 1, True), (5, 64, 64, 64, True, "FLASH", 128, 1, True),
    (260, 66, 100, 64, False, "FLASH", 128, 1, False), (260, 70, 128, 64, True, "FLASH", 128, 1, True),
    (90, 33, 4096, 64, True, "FLASH", 64, 2, True), (90, 33, 4097, 64, True, "FLASH", 64, 2, False),
    (25, 9, 2900, 64, False, "FLASH_HALF", 64, 8, False), (40, 9, 2900, 64, False, "FLASH_HALF", 64, 6, False),
    (2, 20, 1920, 64, True, "FLASH_HALF", 64, 8, True), (3, 40, 16384, 64, True, "FLASH_HALF", 64, 16, True),
    (2, 70, 8256, 64, True, "FLASH_HALF", 64, 12, False), (270, 40, 200, 64, True, "FLASH_PAIR", 64, 1, False),
    (3, 130, 832, 128, True, "FLASH", 128, 8, True), (3, 40, 8256, 128, True, "FLASH", 128, 16, True),
    (20, 9, 2900, 128, True, "FLASH", 64, 8, False), (6, 4, 128, 64, False, "FLASH_HALF", 64, 1, False),
    (6, 4, 130, 64, False, "DECODE", 4, 1, False), (40, 2, 900, 128, True, "DECODE", 2, 2, True),
    (2, 4, 3100, 128, True, "DECODE", 4, 12, True), (2, 4, 7740, 64, True, "DECODE", 4, 12, True)])
def test_every_variant(gpu, oracle, BH, Sq, Sc, D, append, kernel, block_m, splits, inside):
    import ctypes as C

    from polykernel_amd import _lib, kernels

    plan, fused = _lib.Plan(), C.c_int()
    _lib.check(_lib.load().pk_attention_plan(BH, Sq, Sc, D, int(append), 1, C.byref(plan), C.byref(fused)),
               "pk_attention_plan")
    assert (plan.kernel, plan.block_m, plan.splits, bool(fused.value)) == (getattr(_lib, "PLAN_" + kernel), block_m,
                                                                           splits, inside)
    keys = Sc + Sq if append else Sc
    print(f"variant {kernel} BH{BH} Sq{Sq} Sc{Sc} D{D} append={append}", flush=True)
    q, kn, vn = (synth.normal_bf16((1, BH, Sq, D), 200 + i) for i in range(3))
    kc, vc = (synth.normal_bf16((1, BH, keys, D), 203 + i) for i in range(2))
    if append:
        dk, dv = to_dev(kc), to_dev(vc)
        got = from_dev(kernels.fused_kv_append_attention(to_dev(q), to_dev(kn), to_dev(vn), dk, dv, Sc))
        for cache, new, dev in ((kc, kn, dk), (vc, vn, dv)):
            cache[:, :, Sc:] = new
            assert np.array_equal(from_dev(dev), cache)
    else:
        got = from_dev(kernels.attention_prefill(to_dev(q), to_dev(kc), to_dev(vc), None, True))
    _check(oracle, got, q, kc, vc, True)
