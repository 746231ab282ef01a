"""The built-in choices, by shape alone (CPU: the planners need no device)."""
from __future__ import annotations

import ctypes as C

import pytest

from polykernel_amd import _lib


def gemm_plan(M, N, Kd, epi=0, scratch=64 << 20):
    p = _lib.Plan()
    _lib.check(_lib.load().pk_gemm_plan(epi, M, N, Kd, scratch, C.byref(p)), "pk_gemm_plan")
    return p


@pytest.mark.parametrize("M,Kd,N,stream", [(32, 1 << 26, 8, False), (64, 1 << 25, 8, False), (17, 126400000, 8, False),
                                           (64, 33554440, 16, False), (16, 1 << 26, 8, False), (15, 1 << 26, 8, True),
                                           (64, (1 << 24) - 8, 8, True), (1, 126400000, 8, True)])
def test_stream_kernel_holds_a_in_32_bits(M, Kd, N, stream):
    """The streaming kernel addresses A through a 32-bit descriptor and lane
    offsets: A of 2^31 bytes or more keeps the tile kernel."""
    for scratch in (0, 64 << 20):
        assert gemm_plan(M, N, Kd, scratch=scratch).kernel == (_lib.PLAN_STREAM if stream else _lib.PLAN_TILE)
