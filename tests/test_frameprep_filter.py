"""The vertical chroma filter has the form that the frame-prep kernels take as
arguments: at most 8 taps, and at every even height one filter row for all
chroma rows but the first two and the last two, starting at source row 2k - 3
(heights with at most five chroma rows are covered by those five rows)."""
import nes_amd as N
import numpy as np
import pytest


@pytest.mark.parametrize("heights", [range(2, 402, 2), (480, 720, 1080, 1600, 2208, 4320, 8190, 8192, 16384)])
def test_filter_rows_are_uniform_inside(heights):
    inner = None
    for h in heights:
        coef, pos = N.vchroma_filter(h)
        ch, taps = coef.shape
        assert ch == h // 2 and taps <= 8
        for k in range(2, ch - 2):
            assert taps == 8 and pos[k] == 2 * k - 3
            if inner is None:
                inner = coef[k]
            assert np.array_equal(coef[k], inner)
        # no tap reaches past the frame with weight
        for k in range(ch):
            assert pos[k] >= 0 and not coef[k][np.arange(taps) + pos[k] >= h].any()
