"""The projection's front end at 512 and 1024 points, whose last lane butterflies turn signs from transform to transform: any number of
stages against the oracle's scalar butterflies, bit for bit."""
import numpy as np
import pytest

import oracle
from tests import _cabi as cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("H,R,T", [(512, 2, 128), (300, 1, 64), (1024, 1, 128), (772, 2, 256), (513, 1, 5)])
def test_any_number_of_stages(H, R, T, J):
    D = 512 if H <= 512 else 1024
    rng = np.random.RandomState(H + J)
    x = rng.randn(37, H).astype(np.float32)
    x[5] = 0                                            # zeros of either sign
    w = (rng.randn(R, J, D) / np.sqrt(D)).astype(np.float32)
    b = (0.05 * rng.randn(T * 8)).astype(np.float32)
    z = oracle.projection(x, w.reshape(R, J, D, 1, 1), b, T * 8, np.float32(0.7))
    code, score, z_got = cabi.project_hash(x, w, b, T, decay=0.7)
    assert np.array_equal(z_got, z)
    code_o, score_o = oracle.code_score(z.reshape(len(x), T, 8))
    assert np.array_equal(code, code_o)
    np.testing.assert_allclose(score, score_o, rtol=2e-6)
