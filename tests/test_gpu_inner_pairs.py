"""The score gradient where a workgroup takes one table pair, against float64: an fp32 sum of Do products is within Do * 2^-24 of the sum
of their magnitudes."""
import numpy as np
import pytest
import torch

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


# 128 to 191 workgroups of one pair, where tiles that are hardly filled, small tables and wide rows go to the other kernels and the rest
# does not: either side of each line, and either side of 192 workgroups
@pytest.mark.parametrize("B,T,Do", [(1026, 128, 512), (2047, 128, 512), (1700, 128, 64), (1537, 128, 320), (520, 256, 896), (520, 256, 832),
                                    (3073, 64, 256), (3073, 64, 384), (5100, 64, 384), (3073, 64, 960), (3073, 64, 1024), (3072, 96, 1024),
                                    (3072, 126, 384), (3073, 96, 256)])
def test_inner_where_one_table_pair_a_workgroup_may_pay(B, T, Do):
    rng = np.random.RandomState(B + T)
    tables, g = rng.randn(T, 256, Do).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    code = rng.randint(0, 256, size=(B, T)).astype(np.int32)
    got = cabi.lookup_inner(code, g, tables)
    for t in range(T):
        rows = tables[t, code[:, t]].astype(np.float64)
        want, bound = (rows * g).sum(1), (np.abs(rows) * np.abs(g)).sum(1) * Do * 2.0 ** -24
        assert (np.abs(got[:, t] - want) <= bound).all()


# the pairs of an XCD go round the slices from one of their own: slices that are fewer than the XCDs, no multiple of them, more; one pair and two a workgroup
@pytest.mark.parametrize("B,T,Do", [(8000, 64, 64), (7173, 64, 320), (4096, 128, 576), (2100, 200, 832), (3000, 250, 1088)])
def test_inner_goes_round_every_slice(B, T, Do):
    rng = np.random.RandomState(B + Do)
    tables, g = rng.randn(T, 256, Do).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    code = rng.randint(0, 256, size=(B, T)).astype(np.int32)
    got = cabi.lookup_inner(code, g, tables)
    for t in range(0, T, 7):
        rows = tables[t, code[:, t]].astype(np.float64)
        want, bound = (rows * g).sum(1), (np.abs(rows) * np.abs(g)).sum(1) * Do * 2.0 ** -24
        assert (np.abs(got[:, t] - want) <= bound).all()


# the batch cut into launches of 16384 tokens, whose chunks have other numbers of pairs than the whole has
@pytest.mark.parametrize("B,T,Do", [(32768, 32, 512), (32768, 64, 128), (16384 + 4096, 128, 256), (16384, 32, 512), (4096, 128, 512), (3000, 130, 64)])
def test_both_gradients_at_once_have_the_bits_of_the_separate_calls(B, T, Do):
    gen = torch.Generator(device="cuda").manual_seed(B)
    code = torch.randint(0, 256, (B, T), generator=gen, device="cuda", dtype=torch.int32)
    score, g, tables = (torch.randn(*n, generator=gen, device="cuda") for n in ((B, T), (B, Do), (T, 256, Do)))
    code, score, g, tables = (v.cpu().numpy() for v in (code, score, g, tables))
    assert np.array_equal(cabi.lookup_backward(code, score, g, tables, want=(True, False))[0], cabi.lookup_inner(code, g, tables))


# one pair a workgroup and two; the same token everywhere.  Neighbours read the two halves of a row in different orders, by the token's number mod 4
@pytest.mark.parametrize("B,T,Do", [(4096, 128, 512), (8192, 64, 320), (5000, 128, 768), (16384, 32, 256)])
def test_a_token_has_the_same_bits_in_every_tile(B, T, Do):
    rng = np.random.RandomState(T)
    tables, g = rng.randn(T, 256, Do).astype(np.float32), rng.randn(1, Do).astype(np.float32)
    code = rng.randint(0, 256, size=(1, T)).astype(np.int32)
    got = cabi.lookup_inner(code.repeat(B, 0), g.repeat(B, 0), tables)
    assert (got[4:] == got[:-4]).all()
