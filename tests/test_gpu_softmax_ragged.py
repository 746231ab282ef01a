"""Softmax rows whose length is not a multiple of 8 (softmax_ragged_kernel)."""
from __future__ import annotations

import numpy as np
import pytest

from polykernel_amd import metrics as mt
from polykernel_amd import synth
from tests.helpers import f32, from_dev, to_dev

pytestmark = pytest.mark.gpu


# one element up to the longest row, lengths just below and above a change of
# waves or vectors per lane (498 ... 32754 columns), and row counts that leave
# the last chunk of the tensor short or whole; up to 1280 columns with few rows
# (the generic kernel) and with more (the ragged one)
@pytest.mark.parametrize("rows,cols", [(1537, 1), (1539, 3), (1544, 9), (2203, 33), (1903, 101), (2001, 255),
                                       (643, 497), (645, 499), (805, 555), (643, 699),
                                       (323, 1009), (325, 1011), (257, 1279), (1, 1), (5, 3), (8, 9), (3, 497), (6, 499), (7, 1009), (5, 1011), (4, 1521),
                                       (5, 1523), (9, 2033), (5, 2035), (3, 4081), (3, 4083), (5, 8177), (3, 8179),
                                       (3, 16369), (3, 16371), (3, 32753), (2, 32755), (97, 1021)])
def test_softmax_ragged_rows(gpu, oracle, rows, cols):
    from polykernel_amd import kernels

    print(f"ragged softmax {rows}x{cols}", flush=True)
    x = synth.normal_bf16((rows, cols), 170, 2.0)
    lg = synth.normal_f32((rows, cols), 171, 2.0)
    mask = synth.mask_bf16((rows, cols), 172, 0.3)
    mask[:, cols // 2] = 0  # a visible column in every row
    for got, want in ((kernels.softmax(to_dev(x)), oracle.softmax(x)),
                      (kernels.fused_softmax_mask(to_dev(lg), to_dev(mask)), oracle.softmax_mask(lg, mask))):
        # the bars of the vector kernels: sums of exp in another order
        rep = mt.report(from_dev(got), want)
        assert rep.max_ulp <= 1 and (1 - rep.bit_exact) * want.size <= max(2, 0.02 * want.size), rep


@pytest.mark.parametrize("rows", [9, 327])  # the generic kernel, the ragged one
def test_softmax_ragged_neighbour_rows_do_not_mix(gpu, oracle, rows):
    """A row of infinities or NaN between ordinary rows, and a fully masked row:
    only that row's outputs are affected, although its neighbours read its elements."""
    from polykernel_amd import kernels

    cols = 1021
    lg = synth.normal_f32((rows, cols), 173, 2.0)
    mask = synth.mask_bf16((rows, cols), 174, 0.3)
    mask[:, 0] = 0
    lg[2], lg[4, 0], lg[4, -1], lg[6, :] = np.inf, np.nan, np.nan, -np.inf
    mask[7] = 0xFF80
    got = from_dev(kernels.fused_softmax_mask(to_dev(lg), to_dev(mask)))
    want = oracle.softmax_mask(lg, mask)
    assert np.array_equal(np.isnan(f32(got)), np.isnan(f32(want)))
    ok = [0, 1, 3, 5, 8]
    assert not np.isnan(f32(got)[ok]).any()
    rep = mt.report(got[ok], want[ok])
    assert rep.bit_exact >= 0.98 and rep.max_ulp <= 1, rep
