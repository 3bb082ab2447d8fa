"""The table gradient's row sums where their lists can go wrong: tokens around one list and two, a slice that is half a one,
buckets that end at every entry of a step, pieces that one bucket cuts, 512 rows a table.

Bound: an fp32 sum of n products is within n * 2^-24 of the sum of their magnitudes, which is the scale of every element here, and
the result's own rounding 2^-23 of it."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from lookupffn_amd import _lib, ops
from tests import _cabi as cabi

pytestmark = pytest.mark.gpu


def _check(code, w, g, S, accumulate=False):
    B, T = code.shape
    idx = code + (np.arange(T, dtype=np.int32) * S)[None]
    want = oracle.scatter_add(idx, g.astype(np.float64), w.astype(np.float64), T * S).reshape(T, S, -1)
    scale = oracle.scatter_add(idx, np.abs(g).astype(np.float64), np.abs(w).astype(np.float64), T * S).reshape(T, S, -1)
    init = np.random.RandomState(1).randn(*want.shape).astype(np.float32) if accumulate else None
    if accumulate:
        want, scale = want + init, scale + np.abs(init)
    got = cabi.lookup_scatter_sorted(code, w, g, S, accumulate=accumulate, init=init)
    terms = np.bincount(code.ravel(), minlength=S).max() + 1
    assert (np.abs(got - want) <= scale * (terms * 2.0 ** -24 + 2.0 ** -23)).all()
    return got


@pytest.mark.parametrize("B,T,S,Do", [(8192, 3, 256, 64), (8193, 2, 256, 96), (8200, 3, 512, 32), (9217, 2, 16, 160), (15871, 2, 256, 64),
                                      (16384, 9, 1, 32), (16384 + 8193, 2, 256, 96), (37, 3, 256, 32), (513, 2, 8, 608)])
@pytest.mark.parametrize("skew", [False, True])
def test_tokens_around_one_list_and_two(B, T, S, Do, skew):
    rng = np.random.RandomState(B + S + Do)
    code = (rng.zipf(1.2, size=(B, T)) % S if skew else rng.randint(0, S, size=(B, T))).astype(np.int32)
    w, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    got = _check(code, w, g, S)
    assert np.array_equal(got, cabi.lookup_scatter_sorted(code, w, g, S))        # fixed order of additions
    _check(code, w, g, S, accumulate=True)


@pytest.mark.parametrize("lengths", [(1, 2, 3, 4, 5, 6, 7, 8), (1, 1, 1, 1, 1, 1, 1, 60), (63, 64, 65, 0, 0, 1, 0, 3), (0, 0, 700, 0, 1, 0, 0, 0)])
def test_bucket_ends_at_every_entry(lengths):
    rng = np.random.RandomState(sum(lengths))
    code = np.repeat(np.arange(8), lengths).astype(np.int32)[:, None]
    code = np.concatenate([code, rng.permutation(code)], 1)
    _check(code, rng.randn(*code.shape).astype(np.float32), rng.randn(len(code), 96).astype(np.float32), 8)


def test_infinite_gradient_stays_in_its_row():
    rng = np.random.RandomState(5)
    B, T, S, Do = 9000, 2, 256, 96
    code = rng.randint(0, S, size=(B, T)).astype(np.int32)
    code[code == 17] = 18
    code[8500, 0] = 17                                      # alone in its bucket, amid others in its step
    w, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    g[8500] = np.inf
    got = cabi.lookup_scatter_sorted(code, w, g, S)
    assert np.isinf(got[0, 17]).all() and np.isinf(got[1, code[8500, 1]]).all()
    got[0, 17] = got[1, code[8500, 1]] = 0
    assert np.isfinite(got).all()


@pytest.mark.parametrize("B,I,rows,in_tables", [(8193, 8, 1948, 1.0), (9300, 8, 1948, 0.9), (16384, 4, 924, 0.0), (24600, 4, 924, 1.0),
                                                (9000, 4, 5000, 0.0)])      # the last: few pairs a row, one list
def test_flat_rows_of_two_lists(B, I, rows, in_tables):
    rng = np.random.RandomState(B)
    Dv = 96
    idx = rng.randint(0, 256, size=(B, I)) + 256 * np.arange(I)[None]
    idx = np.where(rng.rand(B, I) < in_tables, idx, rng.randint(0, rows, size=(B, I))).clip(0, rows - 1).astype(np.int32)
    w, g = rng.randn(B, I).astype(np.float32), rng.randn(B, Dv).astype(np.float32)
    size = ctypes.c_int64()
    assert _lib.load().lffn_scatter_rows_workspace_bytes(B, I, rows, Dv, ctypes.byref(size)) == 0 and size.value > 0
    idd, gd, wd = (torch.from_numpy(v).cuda() for v in (idx, g, w))
    ws, out = torch.full((size.value,), 0x7f, dtype=torch.uint8, device="cuda"), torch.full((rows, Dv), float("nan"), device="cuda")
    assert _lib.load().lffn_scatter_rows(idd.data_ptr(), gd.data_ptr(), wd.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, I, rows, Dv,
                                         0, 0, _lib.stream_of(gd)) == 0
    got = out.cpu().numpy()
    want = oracle.scatter_add(idx, g.astype(np.float64), w.astype(np.float64), rows)
    scale = oracle.scatter_add(idx, np.abs(g).astype(np.float64), np.abs(w).astype(np.float64), rows)
    terms = np.bincount(idx.ravel()).max()
    assert (np.abs(got - want) <= scale * (terms * 2.0 ** -24 + 2.0 ** -23)).all()


@pytest.mark.parametrize("B,T,Do", [(2049, 64, 384), (3001, 33, 512), (8193, 32, 256), (16384, 33, 128)])
def test_calls_that_had_double_sums_keep_them(B, T, Do):
    """Rounded once, a number is off by 2^-24 / 3^0.5 of its power of two, root mean square; the rows cut by pieces a few roundings more."""
    assert ops.lookup_backward_is_fused(B, T, 256, Do) and B * T * Do < ops.DOUBLE_SCATTER_WORK
    gen = torch.Generator(device="cuda").manual_seed(B)
    code = torch.randint(0, 256, (B, T), generator=gen, device="cuda", dtype=torch.int32)
    score, g = torch.rand(B, T, generator=gen, device="cuda"), torch.randn(B, Do, generator=gen, device="cuda")
    tables = torch.randn(T, 256, Do, generator=gen, device="cuda")
    grad_score, grad = ops._lookup_backward_impl(code, score, g, tables)
    for t in (0, T - 1):
        want = torch.zeros(256, Do, dtype=torch.float64, device="cuda").index_add_(0, code[:, t].long(), score[:, t, None].double() * g.double())
        assert (grad[t] - want).norm() <= 2.0 ** -24 / 3 ** 0.5 * 1.1 * want.norm()
        want = (tables[t].double()[code[:, t].long()] * g.double()).sum(1)
        assert ((grad_score[:, t] - want).abs() <= Do * 2.0 ** -24 * (tables[t].abs()[code[:, t].long()] * g.abs()).sum(1)).all()


@pytest.mark.parametrize("B,T,Do", [(2049, 2, 64), (4096, 2, 128), (9001, 2, 96), (16384, 1, 64)])
@pytest.mark.parametrize("codes", ["one row", "a tenth", "zipf", "even"])
@pytest.mark.parametrize("accumulate", [False, True])
def test_double_sums_are_rounded_once(B, T, Do, codes, accumulate):
    """However many pieces a row's tokens are in: products of two fp32 numbers are exact in a double, n additions are within n * 2^-53 of the
    sum of magnitudes, and there is one rounding to fp32, or two with what is added to."""
    rng = np.random.RandomState(B + len(codes))
    code = {"one row": lambda: np.full((B, T), 77), "a tenth": lambda: np.where(rng.rand(B, T) < 0.1, 77, rng.randint(0, 256, (B, T))),
            "zipf": lambda: (rng.zipf(1.1, (B, T)) - 1) % 256, "even": lambda: rng.randint(0, 256, (B, T))}[codes]().astype(np.int32)
    w, g = rng.rand(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    init = rng.randn(T, 256, Do).astype(np.float32) if accumulate else None
    got = cabi.lookup_scatter_sorted(code, w, g, 256, accumulate=accumulate, init=init).astype(np.float64)
    for t in range(T):
        rows = np.zeros((256, B))
        rows[code[:, t], np.arange(B)] = w[:, t]
        want, scale = rows @ g.astype(np.float64), rows @ np.abs(g).astype(np.float64)
        bound = 2.0 ** -24 * np.abs(want) + np.bincount(code[:, t], minlength=256)[:, None] * 2.0 ** -52 * scale
        if accumulate:
            want = init[t] + want
            bound += 2.0 ** -24 * (np.abs(want) + bound)
        assert (np.abs(got[t] - want) <= bound).all()


@pytest.mark.parametrize("B,T,S,Do", [(40, 2, 256, 96), (3000, 2, 512, 64), (9000, 2, 256, 64), (16384 + 50, 2, 256, 32)])
def test_rows_without_tokens_stay_as_they_are(B, T, S, Do):
    """Added to, a row that no token of the call points at keeps its bits: negative zeros, and numbers that are none."""
    rng = np.random.RandomState(B)
    code = rng.randint(0, S // 4, (B, T)).astype(np.int32) * 4
    code[B // 2:] = np.where(code[B // 2:] == 16, 20, code[B // 2:])       # row 16: in the first list only (row 24 is in no list of table 1)
    code[:, 1] = np.where(code[:, 1] == 24, 28, code[:, 1])
    w, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    init = np.where(np.arange(S)[None, :, None] % 8 < 4, np.float32(-0.0), np.float32("nan")) * np.ones((T, S, Do), np.float32)
    got = cabi.lookup_scatter_sorted(code, w, g, S, accumulate=True, init=init)
    for t in range(T):
        untouched = np.bincount(code[:, t], minlength=S) == 0
        assert untouched.sum() >= S // 2 and np.array_equal(got[t, untouched].view(np.uint32), init[t, untouched].view(np.uint32))
        assert not np.signbit(got[t, ~untouched]).all()


def test_flat_rows_without_tokens_stay_as_they_are():
    rng = np.random.RandomState(7)
    B, I, rows, Dv = 9000, 4, 1500, 96
    idx = (rng.randint(0, rows // 3, (B, I)) * 3).astype(np.int32)
    idd, gd, wd = torch.from_numpy(idx).cuda(), torch.randn(B, Dv, device="cuda"), torch.rand(B, I, device="cuda")
    size = ctypes.c_int64()
    assert _lib.load().lffn_scatter_rows_workspace_bytes(B, I, rows, Dv, ctypes.byref(size)) == 0 and size.value > 0
    ws, out = torch.full((size.value,), 0x7f, dtype=torch.uint8, device="cuda"), torch.full((rows, Dv), -0.0, device="cuda")
    assert _lib.load().lffn_scatter_rows(idd.data_ptr(), gd.data_ptr(), wd.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, I, rows, Dv,
                                         0, 1, _lib.stream_of(gd)) == 0
    untouched = np.bincount(idx.ravel(), minlength=rows) == 0
    got = out.cpu().numpy()
    assert (got[untouched].view(np.uint32) == 0x80000000).all() and (got[~untouched] != 0).any(1).all()


def _rows_within(code, w, g, S, got, init=None, doubles=False):
    """Every row of `got` against float64.  Doubles are rounded once, or twice with what is added to.  An fp32 sum goes through no longer chain than an eighth of its
    row's tokens, or of those in a piece (an eighth of a list of at most 8192, by entries and six for every row), and some twenty additions of parts, lists and launches:
    one lost or doubled pair of a row of 16384 is more than that."""
    B, T = code.shape
    code, w, g = (torch.from_numpy(v).cuda() for v in (code, w, g))
    for t in range(T):
        rows = code[:, t].long()
        want, scale = (torch.zeros(S, g.shape[1], dtype=torch.float64, device="cuda").index_add_(0, rows, a.double()[:, t, None] * b.double())
                       for a, b in ((w, g), (w.abs(), g.abs())))
        n = torch.bincount(rows, minlength=S)[:, None].double()
        if doubles:
            bound = 2.0 ** -24 * want.abs() + n * 2.0 ** -52 * scale
        else:
            bound = (n.clamp(max=(8192 + 6 * S) / 8 + 8) / 8 + 20) * 2.0 ** -24 * scale
        if init is not None:
            want = want + torch.from_numpy(init[t]).cuda().double()
            bound = bound + 2.0 ** -24 * (want.abs() + bound) * (1 if doubles else 4)
        off = (torch.from_numpy(got[t]).cuda().double() - want).abs() - bound
        assert off.max() <= 0, (t, off.argmax() // g.shape[1], off.max())


# pieces are cut by what rows cost: rows of one token each, of none but one, shrinking ones, the many in the last row, fewer tokens than rows
@pytest.mark.parametrize("n", [24, 200, 1000, 8192, 8193, 16384])
@pytest.mark.parametrize("S", [2, 8, 256, 512])
@pytest.mark.parametrize("doubles", [False, True])
def test_pieces_of_skewed_rows(n, S, doubles):
    rng = np.random.RandomState(n + S)
    shrinking = np.minimum((rng.exponential(size=n) * S / 12).astype(int), S - 1)
    spread = np.arange(n) % S
    last = np.where(np.arange(n) < min(n // 4, S - 1), spread, S - 1)
    one = np.full(n, S // 2)
    code = np.stack([shrinking, S - 1 - shrinking, spread, rng.permutation(last), one], 1).astype(np.int32)
    if not doubles:                                         # behind 16384 tokens, so that these are a launch of their own, in fp32
        code = np.concatenate([rng.randint(0, S, (16384, 5)).astype(np.int32), code])
    w, g = rng.randn(*code.shape).astype(np.float32), rng.randn(len(code), 96).astype(np.float32)
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S), doubles=doubles)


# a table's rows are two workgroups' or more: 512 rows; fewer tables x columns than compute units, or up to one and a half times as many.  Either side of each line, and
# rows with more tokens than a part's share, so that parts have one row or none
@pytest.mark.parametrize("B,T,S,Do", [(3000, 65, 512, 256), (3000, 31, 512, 256), (2500, 31, 256, 512), (2500, 32, 256, 512), (2500, 33, 256, 512), (2500, 48, 256, 512),
                                      (2500, 49, 256, 512), (2100, 5, 64, 96), (2100, 5, 32, 64), (16384 + 2500, 31, 256, 512), (16384 + 9000, 33, 256, 480),
                                      (16384 + 700, 9, 512, 224)])
def test_rows_of_several_workgroups(B, T, S, Do):
    rng = np.random.RandomState(B + T + S)
    code = rng.randint(0, S, (B, T))
    code[:, 0] = S - 1                                      # one row has all
    code[:, 1] = np.where(rng.rand(B) < 0.6, S // 2, code[:, 1])
    code[:, 2] = np.minimum(rng.exponential(size=B) * S / 12, S - 1)
    code[:, 3] = np.where(np.arange(B) < B // 2, 0, S - 1)      # and in either list another
    code = code.astype(np.int32)
    w, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    got = cabi.lookup_scatter_sorted(code, w, g, S)
    _rows_within(code, w, g, S, got, doubles=B <= 16384)
    assert np.array_equal(got, cabi.lookup_scatter_sorted(code, w, g, S))
    init = rng.randn(T, S, Do).astype(np.float32)
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S, accumulate=True, init=init), init=init, doubles=B <= 16384)
