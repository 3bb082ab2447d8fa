"""The sorted accumulation on top of what the rows hold: the sums are those of the plain call, added once, and rows that no token
points at are not touched."""
import numpy as np
import pytest

from tests import _cabi as cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,S,Do,skew", [(1, 2, 4, 64, False), (300, 1, 2, 64, False), (500, 4, 512, 96, True),
                                           (2100, 3, 256, 288, True), (5000, 2, 256, 32, False), (16384, 1, 256, 64, True)])
def test_sorted_scatter_adds_each_row_once(B, T, S, Do, skew):
    rng = np.random.RandomState(B + S)
    code = rng.randint(0, S, size=(B, T))
    if skew:                                            # most tokens on one row, whose list every wavefront has a piece of
        code[rng.rand(B, T) < 0.9] = S // 2
    code[code == S - 1] = 0                             # and one row that is nobody's
    code = code.astype(np.int32)
    score = rng.rand(B, T).astype(np.float32)
    g = rng.randn(B, Do).astype(np.float32)
    plain = cabi.lookup_scatter_sorted(code, score, g, S)
    init = rng.randn(T, S, Do).astype(np.float32)
    init[:, S - 1] = np.nan
    got = cabi.lookup_scatter_sorted(code, score, g, S, accumulate=True, init=init)
    assert np.isnan(got[:, S - 1]).all()
    assert np.array_equal(got[:, :S - 1], (init + plain)[:, :S - 1])
