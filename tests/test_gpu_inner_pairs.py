"""The score gradient where a workgroup takes one table pair, against float64: an fp32 sum of Do products is within Do * 2^-24 of the sum
of their magnitudes."""
import numpy as np
import pytest

from tests import _cabi as cabi

pytestmark = pytest.mark.gpu


# around the lines between one pair, two and the other kernels: workgroups of one pair 126, 128, 192, 256, 260; short last tiles
@pytest.mark.parametrize("B,T,Do", [(2048, 126, 64), (1025, 128, 64), (3073, 64, 128), (2049, 128, 192), (6145, 32, 64),
                                    (4096, 128, 64), (16000, 32, 64), (4097, 104, 64)])
def test_inner_of_one_table_pair_a_workgroup(B, T, Do):
    S = 256
    rng = np.random.RandomState(B + T)
    tables = rng.randn(T, S, Do).astype(np.float32)
    code = rng.randint(0, S, size=(B, T)).astype(np.int32)
    g = rng.randn(B, Do).astype(np.float32)
    got = cabi.lookup_inner(code, g, tables)
    for t in range(T):
        rows = tables[t, code[:, t]].astype(np.float64)
        want, bound = (rows * g).sum(1), (np.abs(rows) * np.abs(g)).sum(1) * Do * 2.0 ** -24
        assert (np.abs(got[:, t] - want) <= bound).all()
    assert np.array_equal(got, cabi.lookup_inner(code, g, tables))      # one owner a sum
