"""The table gradient's row sums where their lists can go wrong: tokens around one list and two, a slice that is half a one,
buckets that end at every entry of a step, pieces that one bucket cuts, 512 rows a table, rows of several workgroups.

Up to 16384 tokens and 4e8 products the sums are doubles and their tokens one list; of other calls every 16384 tokens are one list or two, in fp32.  Small calls
in fp32 are the end of one of more than 16384 tokens, whose last launch has the tokens in question and adds to the rows of the first."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from lookupffn_amd import _lib, ops
from tests import _cabi as cabi

pytestmark = pytest.mark.gpu


def _in_doubles(B, T, Do):
    return B <= ops.SCATTER_CHUNK_TOKENS and B * T * Do < ops.DOUBLE_SCATTER_WORK


def _bound(want, scale, n, piece, doubles):
    """How far a row of n tokens may be off.  Doubles are rounded once.  An fp32 sum goes through no longer chain than an eighth of its row's tokens, or of those in a
    piece, and some twenty additions of parts, lists and launches: one lost or doubled pair of a row of 16384 is more than that."""
    if doubles:
        return 2.0 ** -24 * want.abs() + n * 2.0 ** -52 * scale
    return (n.clamp(max=piece) / 8 + 20) * 2.0 ** -24 * scale


def _rows_within(code, w, g, S, got, init=None, tables=None):
    """Every row of `got`, or of some of its tables, against float64."""
    B, T = code.shape
    doubles = _in_doubles(B, T, g.shape[1])
    code, w, g = (torch.from_numpy(v).cuda() for v in (code, w, g))
    for t in range(T) if tables is None else tables:
        rows = code[:, t].long()
        weights = torch.zeros(S, B, dtype=torch.float64, device="cuda")
        weights[rows, torch.arange(B, device="cuda")] = w[:, t].double()
        want, scale = weights @ g.double(), weights.abs() @ g.double().abs()
        n = torch.bincount(rows, minlength=S)[:, None].double()
        bound = _bound(want, scale, n, (8192 + 6 * S) / 8 + 8, doubles)      # a list of at most 8192 in eight pieces, by entries and six for every row
        if init is not None:                                # each launch that adds rounds once more
            want = want + torch.from_numpy(init[t]).cuda().double()
            bound = bound + 2.0 ** -24 * (want.abs() + bound) + (0 if doubles else (B // 16384 + 1) * 2.0 ** -24 * (scale + want.abs()))
        off = (torch.from_numpy(got[t]).cuda().double() - want).abs() - bound
        assert off.max() <= 0, (t, off.argmax() // g.shape[1], off.max())


def _behind(rng, code, S, fp32):
    """`code` alone, or behind 16384 tokens of a launch of their own."""
    return np.concatenate([rng.randint(0, S, (16384, code.shape[1])), code]).astype(np.int32) if fp32 else code.astype(np.int32)


@pytest.mark.parametrize("n,T,S,Do", [(4500, 2, 256, 96), (8192, 3, 256, 64), (8193, 2, 256, 96), (8200, 3, 512, 32), (9217, 2, 16, 160), (15871, 2, 256, 64),
                                      (16384, 9, 1, 32), (37, 3, 256, 32), (513, 2, 8, 608)])
@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("fp32", [False, True])
def test_tokens_around_one_list_and_two(n, T, S, Do, skew, fp32):
    rng = np.random.RandomState(n + S + Do)
    code = _behind(rng, rng.zipf(1.2, size=(n, T)) % S if skew else rng.randint(0, S, size=(n, T)), S, fp32)
    B = len(code)
    assert _in_doubles(B, T, Do) != fp32
    w, g, init = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32), rng.randn(T, S, Do).astype(np.float32)
    got = cabi.lookup_scatter_sorted(code, w, g, S)
    _rows_within(code, w, g, S, got)
    assert np.array_equal(got, cabi.lookup_scatter_sorted(code, w, g, S))        # fixed order of additions
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S, accumulate=True, init=init), init=init)


# one list and two in fp32 that overwrite, as a call's first launch does
@pytest.mark.parametrize("B,T,S,Do", [(4500, 128, 256, 768), (8193, 64, 256, 768), (9217, 64, 512, 704), (15871, 64, 16, 416), (16384, 65, 1, 384)])
def test_lists_of_a_first_launch_in_fp32(B, T, S, Do):
    assert not _in_doubles(B, T, Do)
    rng = np.random.RandomState(B)
    code, w, g = rng.randint(0, S, (B, T)).astype(np.int32), rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    code[:, 1] = S - 1
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S), tables=(0, 1, T // 2, T - 1))


@pytest.mark.parametrize("lengths", [(1, 2, 3, 4, 5, 6, 7, 8), (1, 1, 1, 1, 1, 1, 1, 60), (63, 64, 65, 0, 0, 1, 0, 3), (0, 0, 700, 0, 1, 0, 0, 0)])
@pytest.mark.parametrize("fp32", [False, True])
def test_bucket_ends_at_every_entry(lengths, fp32):
    rng = np.random.RandomState(sum(lengths))
    code = np.repeat(np.arange(8), lengths)[:, None]
    code = _behind(rng, np.concatenate([code, rng.permutation(code)], 1), 8, fp32)
    w, g = rng.randn(*code.shape).astype(np.float32), rng.randn(len(code), 96).astype(np.float32)
    assert _in_doubles(len(code), 2, 96) != fp32
    _rows_within(code, w, g, 8, cabi.lookup_scatter_sorted(code, w, g, 8))


@pytest.mark.parametrize("B", [9000, 16384 + 9000])
def test_infinite_gradient_stays_in_its_row(B):
    rng = np.random.RandomState(5)
    T, S, Do = 2, 256, 96
    code = rng.randint(0, S, size=(B, T)).astype(np.int32)
    code[code == 17] = 18
    code[B - 500, 0] = 17                                     # alone in its bucket, amid others in its step
    w, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    g[B - 500] = np.inf
    got = cabi.lookup_scatter_sorted(code, w, g, S)
    assert np.isinf(got[0, 17]).all() and np.isinf(got[1, code[B - 500, 1]]).all()
    got[0, 17] = got[1, code[B - 500, 1]] = 0
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
    want, scale = (torch.from_numpy(oracle.scatter_add(idx, a.astype(np.float64), b.astype(np.float64), rows)) for a, b in ((g, w), (np.abs(g), np.abs(w))))
    n = torch.from_numpy(np.bincount(idx.ravel(), minlength=rows))[:, None].double()
    assert ((out.cpu().double() - want).abs() <= _bound(want, scale, n, B * I, False)).all()


@pytest.mark.parametrize("B,T,Do", [(2049, 64, 384), (3001, 32, 512), (8193, 32, 256), (16384, 33, 128)])
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


# pieces are cut by what rows cost: rows of one token each, of none but one, shrinking ones, the many in the last row, fewer tokens than rows
@pytest.mark.parametrize("n", [24, 200, 1000, 8192, 8193, 16384])
@pytest.mark.parametrize("S", [2, 8, 256, 512])
@pytest.mark.parametrize("fp32", [False, True])
def test_pieces_of_skewed_rows(n, S, fp32):
    rng = np.random.RandomState(n + S)
    shrinking = np.minimum((rng.exponential(size=n) * S / 12).astype(int), S - 1)
    spread = np.arange(n) % S
    last = np.where(np.arange(n) < min(n // 4, S - 1), spread, S - 1)
    one = np.full(n, S // 2)
    code = np.stack([shrinking, S - 1 - shrinking, spread, rng.permutation(last), one], 1)
    code = _behind(rng, code, S, fp32)
    assert _in_doubles(len(code), 5, 96) != fp32
    w, g = rng.randn(*code.shape).astype(np.float32), rng.randn(len(code), 96).astype(np.float32)
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S))


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
    _rows_within(code, w, g, S, got)
    assert np.array_equal(got, cabi.lookup_scatter_sorted(code, w, g, S))
    init = rng.randn(T, S, Do).astype(np.float32)
    _rows_within(code, w, g, S, cabi.lookup_scatter_sorted(code, w, g, S, accumulate=True, init=init), init=init)
