"""The built-in choices, by shape alone (CPU: the planners need no device)."""
from __future__ import annotations

import ctypes as C

import pytest

from polykernel_amd import _lib


def gemm_plan(M, N, Kd, epi=0, scratch=64 << 20):
    p = _lib.Plan()
    _lib.check(_lib.load().pk_gemm_plan(epi, M, N, Kd, scratch, C.byref(p)), "pk_gemm_plan")
    return p


def int8_plan(M, N, Kd, scratch=16 << 20):
    p = _lib.Plan()
    _lib.check(_lib.load().pk_int8_plan(M, N, Kd, scratch, C.byref(p)), "pk_int8_plan")
    return p


@pytest.mark.parametrize("M,Kd,N,stream", [(32, 1 << 26, 8, False), (64, 1 << 25, 8, False), (17, 126400000, 8, False),
                                           (64, 33554440, 16, False), (16, 1 << 26, 8, False), (15, 1 << 26, 8, True),
                                           (64, (1 << 24) - 8, 8, True), (1, 126400000, 8, True)])
def test_stream_kernel_holds_a_in_32_bits(M, Kd, N, stream):
    """The streaming kernel addresses A through a 32-bit descriptor and lane
    offsets: A of 2^31 bytes or more keeps the tile kernel."""
    for scratch in (0, 64 << 20):
        assert gemm_plan(M, N, Kd, scratch=scratch).kernel == (_lib.PLAN_STREAM if stream else _lib.PLAN_TILE)


# us of tile / ring kernel in a replayed graph, rounded; both sides of every line of the rule
@pytest.mark.parametrize("epi,M,N,Kd,ring", [
    (0, 300, 1024, 128, False), (0, 300, 1024, 768, True),        # 4.0 / 5.0, 10.3 / 8.2
    (0, 85, 16, 256, False), (0, 85, 16, 1024, True),             # 4.4 / 5.4, 9.3 / 8.3
    (1, 700, 512, 64, False), (1, 700, 512, 768, True),           # 5.3 / 6.4, 11.9 / 9.9
    (1, 1555, 16, 512, False), (1, 1555, 16, 1024, True),         # 7.7 / 9.7, 13.1 / 11.9
    (2, 304, 1024, 64, False), (2, 700, 4096, 256, True),         # 4.4 / 5.2, 11.0 / 9.9
    (3, 402, 24, 64, False),                                      # 4.0 / 5.1
    (0, 4000, 1024, 64, False), (1, 4000, 1024, 64, True),        # 4.2 / 4.5, 14.1 / 11.1 (128 x 128)
    (0, 4000, 16384, 8, False), (2, 4000, 4096, 8, True),         # 45.9 / 55, (register-staged 256 x 256)
    (1, 4000, 2304, 256, False), (0, 4000, 2304, 256, True),      # 20.3 / 22.7, 16.4 / 14.6 (direct 256 x 256)
    (1, 10000, 4096, 512, False), (1, 1500, 4096, 512, True),     # 76.6 / 98.8, 22.9 / 19.0
    (0, 777, 12288, 4096, True), (1, 501, 8192, 2048, True), (2, 501, 2048, 8192, True), (0, 4096, 16384, 4096, False)])
def test_gemm_takes_the_faster_kernel(epi, M, N, Kd, ring):
    assert gemm_plan(M, N, Kd, epi).kernel == (_lib.PLAN_RING if ring else _lib.PLAN_TILE)


@pytest.mark.parametrize("epi,M,N,Kd,plan", [
    (2, 64, 16448, 64, (_lib.PLAN_TILE, 64, 64)), (0, 64, 20000, 16, (_lib.PLAN_TILE, 64, 64)),
    (0, 32, 20000, 16, (_lib.PLAN_STREAM, 32, 128)), (0, 64, 20000, 1024, (_lib.PLAN_STREAM, 64, 128)),
    (0, 64, 42496, 4544, (_lib.PLAN_RING, 96, 256)), (0, 40, 50256, 2560, (_lib.PLAN_RING, 96, 256)),
    (0, 32, 50256, 2560, (_lib.PLAN_STREAM, 32, 128)), (0, 64, 16384, 4096, (_lib.PLAN_STREAM, 64, 64))])
def test_few_rows_take_the_faster_kernel(epi, M, N, Kd, plan):
    p = gemm_plan(M, N, Kd, epi, scratch=0)
    assert (p.kernel, p.block_m, p.block_n) == plan


def test_conformance_objects_launch_their_own_gemm():
    """A served RMSNorm -> MatMul call launches the object's pk_gemm only where the
    built-in choice is a tile; the conformance set holds one such shape per staging."""
    from polykernel_amd import emit

    tiles = [s for s in emit.PANEL_SHAPES
             if all(gemm_plan(*s, scratch=n).kernel == _lib.PLAN_TILE for n in (0, 64 << 20))]
    assert {s[1] % 8 == 0 for s in tiles} == {True, False}


@pytest.mark.parametrize("M,N,Kd,odd", [(1, 50257, 8, True), (32, 50257, 8, True), (33, 50257, 56, False),
                                        (33, 50257, 64, True), (64, 8191, 8, True), (65, 50257, 64, False)])
def test_odd_rows_take_the_faster_kernel(M, N, Kd, odd):
    assert gemm_plan(M, N, Kd).kernel == (_lib.PLAN_ODD if odd else _lib.PLAN_TILE)


T, S, R = _lib.PLAN_TILE, _lib.PLAN_STREAM, _lib.PLAN_RING


# us of the column-split stream or generic kernel / of the K-split stream or ring
@pytest.mark.parametrize("M,N,Kd,kernel", [
    (53, 1024, 56, T), (44, 512, 368, T), (39, 8192, 64, T), (224, 2800, 184, T),  # 3.0 / 4.9, 4.1 / 6.8, 3.5 / 5.0, 5.3 / 6.1
    (35, 688, 27968, T), (66, 48, 27144, T),                                       # 23 / 30, 13 / 29
    (108, 128, 512, R), (300, 12288, 4096, R), (64, 12288, 4096, R), (33, 12288, 4096, R), (400, 4096, 1032, R),
    (3, 24640, 32, T), (29, 36064, 64, T), (26, 144, 28280, T),                    # 2.8 / 3.5, 5.8 / 7.2, 14.6 / 17.4
    (3, 4000, 104, S), (32, 30000, 64, S), (16, 16384, 4096, S), (32, 4096, 14336, S), (16, 28672, 8192, T)])
def test_int8_takes_the_faster_kernel(M, N, Kd, kernel):
    assert int8_plan(M, N, Kd).kernel == kernel


# one or two k-steps: rounds that are nearly full; up to 128 columns; few tiles over a long K
@pytest.mark.parametrize("M,N,Kd,ring", [
    (160, 36848, 64, False), (43, 30000, 64, True), (1529, 1984, 64, False), (300, 30000, 64, True),   # 10.9 / 17.1, 7.2 / 5.6
    (556, 128, 8576, True), (120, 400, 23624, False), (60, 128, 8576, False)])                         # 20.3 / 16.0
def test_int8_ring_at_short_k(M, N, Kd, ring):
    assert (int8_plan(M, N, Kd).kernel == _lib.PLAN_RING) == ring


# weights above 32 MB whose rows are a multiple of 1024 bytes: full rounds of workgroups
@pytest.mark.parametrize("M,N,Kd", [(1, 5120, 16384), (1, 3072, 22784), (16, 8192, 8192), (8, 4096, 18944), (1, 20480, 4352),
                                    (16, 6144, 14592), (1, 12288, 7296)])
def test_int8_stream_fills_its_rounds(M, N, Kd):
    p = int8_plan(M, N, Kd)
    units = -(-N // p.block_n) * p.splits
    assert p.kernel == S and (216 <= units <= 256 or 464 <= units <= 512), units


# us of the generic / the ragged kernel: 2.6 / 3.8, 3.0 / 3.7, 3.5 / 3.7, 4.0 / 4.4, 4.7 / 5.2, then the other way
@pytest.mark.parametrize("rows,cols,ragged", [
    (64, 33, False), (1000, 33, False), (512, 300, False), (256, 700, False), (256, 1021, False), (4000, 33, True),
    (2090, 23, False), (2400, 23, True), (655, 555, False), (900, 555, True),   # 3.8 / 4.5, 3.9 / 4.5
    (1000, 300, True), (512, 1021, True), (64, 2047, True), (1, 32753, True), (16336, 1021, True), (16336, 1024, False),
    (1, 32755, False)])
def test_softmax_takes_the_faster_kernel(rows, cols, ragged):
    p = _lib.Plan()
    _lib.check(_lib.load().pk_softmax_plan(rows, cols, C.byref(p)), "pk_softmax_plan")
    assert (p.kernel == _lib.PLAN_RAGGED) == ragged


def attention_plan(BH, S_q, S_cache, D, append=True, causal=True):
    p, fused = _lib.Plan(), C.c_int()
    _lib.check(_lib.load().pk_attention_plan(BH, S_q, S_cache, D, int(append), int(causal), C.byref(p),
                                             C.byref(fused)), "pk_attention_plan")
    return p, bool(fused.value)


# us with as many splits as before / now
@pytest.mark.parametrize("BH,S_q,S_cache,D,append,splits", [
    (160, 1, 4096, 64, False, 1),    # 38 in two rounds / 31
    (100, 4, 4096, 64, False, 2),    # 32 in 4 / 26
    (8, 1, 16384, 128, False, 16), (1, 1, 1 << 20, 128, False, 16),
    (100, 1, 509, 128, True, 1), (100, 2, 1021, 64, True, 1),   # 10.2 in two / 8.6, 11.3 / 10.1
    (32, 1, 256, 128, True, 1), (32, 4, 2048, 128, True, 8), (1, 2, 8, 128, True, 1), (300, 1, 1 << 16, 64, True, 1)])
def test_decode_splits(BH, S_q, S_cache, D, append, splits):
    p, fused = attention_plan(BH, S_q, S_cache, D, append)
    assert (p.kernel, p.splits, fused) == (_lib.PLAN_DECODE, splits, append)
    assert p.splits == 1 or p.splits * BH <= 256


@pytest.mark.parametrize("S_q,S_cache,D,append,decode", [
    (4, 128, 64, False, False), (3, 4, 64, False, False), (4, 129, 64, False, True), (2, 4, 64, False, True),
    (4, 128, 128, False, True), (4, 124, 64, True, True), (5, 4096, 64, False, False), (4, 0, 64, True, True)])
def test_few_queries_on_short_keys(S_q, S_cache, D, append, decode):
    """Three and four queries on up to 128 keys of D 64: flash 5.0 us, decode 5.9 (96 heads, 4 keys)."""
    assert (attention_plan(96, S_q, S_cache, D, append)[0].kernel == _lib.PLAN_DECODE) == decode


# us of the variant that was taken before / of this one
@pytest.mark.parametrize("BH,S_q,S_cache,append,causal,kernel,block_m,splits,inside", [
    (141, 12, 9472, True, True, "FLASH", 64, 1, True),         # half ring 100 / full 71
    (43, 160, 6656, True, True, "FLASH", 64, 1, True),         # 70.3 / 54.0
    (16, 1021, 1021, False, True, "FLASH_HALF", 64, 1, False),  # 14.1 full / 13.2
    (32, 333, 1200, True, True, "FLASH_HALF", 64, 1, False),    # 12 steps, six tiles of a head read the same keys
    (7, 1995, 1995, False, False, "FLASH_HALF", 64, 1, False),  # 32.0 in two / 22.1
    (108, 99, 2816, False, False, "FLASH", 64, 1, False),       # 34.8 half / 27.8
    (7, 37, 64, True, True, "FLASH", 128, 1, True),             # 10.1 append first / 7.5
    (1, 12, 64, True, True, "FLASH", 128, 1, True),             # 7.2 / 6.4
    (1, 12, 192, True, True, "FLASH_HALF", 64, 1, False),       # 128 x 64 appending is 1.06 times as long
    (449, 68, 73, False, True, "FLASH", 128, 1, False),         # pair 16.0 / 13.2
    (466, 74, 128, True, True, "FLASH", 128, 1, True),          # 26.1 / 22.6
    (128, 256, 2048, True, True, "FLASH_PAIR", 64, 1, False), (40, 1024, 1024, False, False, "FLASH_PAIR", 64, 1, False),
    (64, 512, 512, False, True, "FLASH", 128, 1, False),
    (64, 500, 64, True, True, "FLASH", 128, 1, True), (64, 500, 65, True, True, "FLASH_PAIR", 64, 1, False)])  # 21.8 / 19.5
def test_flash_takes_the_faster_variant_at_64(BH, S_q, S_cache, append, causal, kernel, block_m, splits, inside):
    p, fused = attention_plan(BH, S_q, S_cache, 64, append, causal)
    assert (p.kernel, p.block_m, p.splits, fused) == (getattr(_lib, "PLAN_" + kernel), block_m, splits, inside)


@pytest.mark.parametrize("D", [64, 128])
def test_flash_splits_stay_in_one_round(D):
    for BH, S_q, S_cache in ((1, 8, 1 << 17), (8, 500, 0), (16, 7, 1000), (12, 29, 3200), (8, 1000, 24), (40, 64, 8192),
                             (200, 33, 8192), (1, 5, 1 << 20)):
        p, _ = attention_plan(BH, S_q, S_cache, D)
        tiles = BH * -(-S_q // p.block_m)
        assert p.splits == 1 or (tiles * p.splits <= 256 and p.splits < -(-(S_cache + S_q) // p.block_n))
    assert attention_plan(16, 7, 1000, 128)[0].splits > 1 and attention_plan(12, 29, 3200, 128)[0].splits > 1
    assert attention_plan(8, 500, 0, 128)[0].splits == 1       # 15.9 in four / 12.7
    assert attention_plan(6, 5, 11328, 128, False)[0].splits == 16 and attention_plan(1, 60, 5696, 128)[0].splits == 16
    assert attention_plan(4, 16, 8192, 64)[0].splits < 16      # 19.8 in sixteen / 18.3


@pytest.mark.parametrize("M,N,Kd", [(16, 4096, 8192), (1, 4096, 4096), (16, 28672, 8192), (300, 4096, 4096)])
def test_int8_refuses_unaligned_scratch_where_the_column_kernel_splits(M, N, Kd):
    """Scratch that is refused stays refused whichever kernel the product takes
    (nothing is launched: the addresses are made up)."""
    lib, cfg, at = _lib.load(), _lib.Config(), 1 << 20
    assert lib.pk_int8_default_config(M, N, Kd, cfg) == 0 and cfg.block_k < Kd
    for ws, size in ((at + 8, 1 << 28), (at, 64)):
        assert lib.pk_matmul_int8_ex(0, at, at, at, at, None, M, N, Kd, None, ws, size, None) == _lib.PK_ERR_WORKSPACE
