"""64 x 64 blocks on the fp16 matrix cores (csrc/bh4_split.hip) against 64 bits."""
import math

import pytest
import torch

from lookupffn_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV)


def _hadamard(n):
    h = torch.ones(1, 1, dtype=torch.float64)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _blocks(w, u):
    n, D = u.shape
    return torch.matmul(w.contiguous().unsqueeze(0), u.reshape(n, D // 64, 64, 1)).reshape(n, D)


def _rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


# Four stages of sums over 64: a product is off by 2^-22 at most, a sum by 2^-24 in each of 6 instructions; then butterflies, log2 D
# additions.  Per stage 2^-22 + sqrt(6 + 4) 2^-24 at worst, of either sign from stage to stage: 2 * 4.3e-7.
REL = 8.6e-7


# every number of blocks, both forms of the kernel (few and many workgroups), rows around the 16 of a tile, columns short of D, codes
# short of them
@pytest.mark.parametrize("B,H,D,R,T", [(1, 64, 64, 2, 16), (33, 100, 128, 2, 30), (70, 256, 256, 1, 32), (4200, 200, 256, 1, 32),
                                       (31, 512, 512, 2, 100), (2300, 500, 512, 2, 128), (17, 768, 1024, 1, 128), (4100, 1024, 1024, 1, 128)])
@pytest.mark.parametrize("with_ln", [True, False])
def test_against_64_bits(B, H, D, R, T, with_ln):
    gen = torch.Generator(device=DEV).manual_seed(B + D)
    J, NB = 4, D // 64
    x, w = 1.5 * _randn(gen, B, H) + 0.3, _randn(gen, R, J, NB, 64, 64) / math.sqrt(64 * D)
    lw, lb = (1 + 0.1 * _randn(gen, H), 0.1 * _randn(gen, H)) if with_ln else (None, None)
    bias = 0.05 * _randn(gen, T * 8) if with_ln else None
    split = ops.bh4_fold_split(w, False)
    codes, scores = ops.bh4_block_front(x, lw, lb, 1e-5, split, R, J, D, bias, T, 0.7, 0.3)
    few = min(B, 20)
    for a, b in zip(ops.bh4_block_front(x[:few], lw, lb, 1e-5, split, R, J, D, bias, T, 0.7, 0.3), (codes, scores)):
        assert torch.equal(a, b[:few])                # whichever form, whatever the neighbours
    some = list(range(min(B, 40))) + [B - 1]
    h = x[some].double().cpu()
    if with_ln:
        h = torch.nn.functional.layer_norm(h, (H,), lw.double().cpu(), lb.double().cpu(), 1e-5)
    h = torch.cat([h, torch.zeros(len(some), D - H, dtype=torch.float64)], 1)
    w64, HD, HN = w.double().cpu(), _hadamard(D), _hadamard(NB)
    z = []
    for r in range(R):
        u = h
        for j in range(J):
            u = _blocks(w64[r, j], u) @ HD
        z.append(0.7 * u + 0.3 * h)
    z = torch.cat(z, 1)[:, :T * 8] + (bias.double().cpu() if with_ln else 0)
    z8, size = z.view(len(some), T, 8), z.pow(2).mean().sqrt()
    code = ((z8 > 0) * (2 ** torch.arange(7, -1, -1))).sum(-1)
    same = code == codes[some].cpu()
    # six standard deviations of an error of REL (and LayerNorm's, as large)
    assert (z8.abs().amin(-1)[~same] <= 12 * REL * size).all() and same.double().mean() >= 0.999
    score = z8.abs().sum(-1) / (1 + torch.exp(-2 * z8.abs())).prod(-1)
    # a score moves at most 2.2 times as far as a z of its eight (1 + 1.25 sum / product for small ones), 8^0.5 of them together
    assert ((scores[some].double().cpu() - score)[same].norm() / score.norm()) <= 6.3 * 2 * REL

    g_z = _randn(gen, B, T * 8)
    split_t = ops.bh4_fold_split(w, True)
    g_x, stage_g = ops.bh4_block_bwd_split(g_z, split_t, R, J, D, H, 0.7, 0.3)
    g_few, stage_few = ops.bh4_block_bwd_split(g_z[:few], split_t, R, J, D, H, 0.7, 0.3)
    assert torch.equal(g_few, g_x[:, :few]) and torch.equal(stage_few, stage_g[:, :, :few])
    g_pad = torch.cat([g_z[some].double().cpu(), torch.zeros(len(some), R * D - T * 8, dtype=torch.float64)], 1)
    for r in range(R):
        g = g_pad[:, r * D:(r + 1) * D]
        G = 0.7 * g
        for j in range(J - 1, -1, -1):
            assert _rel(stage_g[r, j][some], torch.matmul(HN, G.view(-1, NB, 64)).reshape(-1, D)) <= REL
            G = _blocks(w64[r, j].transpose(-1, -2), G @ HD)
        assert _rel(g_x[r][some], (G + 0.3 * g)[:, :H]) <= REL


@pytest.mark.parametrize("B,H,D,R,T", [(1, 64, 64, 2, 16), (33, 100, 128, 2, 29), (70, 256, 256, 1, 32), (4200, 200, 256, 1, 31),
                                       (31, 512, 512, 2, 100), (2300, 500, 512, 2, 128), (17, 768, 1024, 1, 127), (4100, 1024, 1024, 1, 128)])
def test_backward_from_scores(B, H, D, R, T):
    """The scores' derivative inside the kernel: what code_score_bwd and the backward from its result give, bit for bit; the bias's
    gradient, sums of sixteen and then of at most 256 numbers and chunks, within that many roundings of their magnitudes."""
    gen = torch.Generator(device=DEV).manual_seed(B + T)
    J = 4
    split_t = ops.bh4_fold_split(_randn(gen, R, J, D // 64, 64, 64) / math.sqrt(64 * D), True)
    z, g_score = 2 * _randn(gen, B, T * 8), _randn(gen, B, T)
    z[0, :8] = 0
    z[-1, ::3] *= 1e-8
    g_z = ops.code_score_bwd(z.view(B, T, 8), g_score).view(B, T * 8)
    g_x, stage_g, g_bias = ops.bh4_block_score_bwd_split(z, g_score, split_t, R, J, D, H, 0.7, 0.3, True)
    want_x, want_stage = ops.bh4_block_bwd_split(g_z, split_t, R, J, D, H, 0.7, 0.3)
    assert torch.equal(g_x, want_x) and torch.equal(stage_g, want_stage)
    assert ((g_bias - g_z.double().sum(0)).abs() <= 64 * 2.0 ** -24 * g_z.double().abs().sum(0)).all()
    assert ops.bh4_block_score_bwd_split(z, g_score, split_t, R, J, D, H, 0.7, 0.3, False)[2].numel() == 0
    for n in (4, 100004, 3 << 20):                    # and the array that it clears, to its last number and no further
        clear = torch.ones(n + 4, device=DEV)
        rc = _lib.load().lffn_bh4_block_score_bwd_split_f32(z.data_ptr(), g_score.data_ptr(), split_t.data_ptr(), g_x.data_ptr(), stage_g.data_ptr(),
                                                            None, clear.data_ptr(), n, B, H, D, R, J, T, 64, 0.7, 0.3, _lib.stream_of(z))
        assert rc == 0 and not clear[:n].any() and clear[n:].all()


@pytest.mark.parametrize("n", [0, 4, 1000, 3 << 20])
def test_backward_of_no_tokens_clears(n):
    clear = torch.ones(n + 4, device=DEV)
    args = (0, 256, 256, 1, 4, 32, 64, 0.7, 0.3, _lib.stream_of(clear))
    entry = _lib.load().lffn_bh4_block_score_bwd_split_f32
    assert entry(None, None, None, None, None, None, None, 0, *args) == 0
    assert entry(None, None, None, None, None, None, clear.data_ptr(), n, *args) == 0 and not clear[:n].any() and clear[n:].all()


@pytest.mark.parametrize("stages,NB", [(1, 1), (3, 2), (8, 8), (4, 16)])
def test_both_foldings_in_one_launch(stages, NB):
    w = torch.randn(stages, 1, NB, 64, 64, device=DEV)
    want = [ops.bh4_fold_split(w, t) for t in (False, True)]
    got = [torch.full_like(s, float("nan")) for s in want]
    assert _lib.load().lffn_bh4_fold_split_both_f32(w.data_ptr(), got[0].data_ptr(), got[1].data_ptr(), stages, NB, 64, _lib.stream_of(w)) == 0
    assert all(torch.equal(a.view(torch.int32), b.view(torch.int32)) for a, b in zip(got, want))


# both forms of the kernel (few and many workgroups), rows around the 16 of a tile, columns short of D, codes short of them
@pytest.mark.parametrize("B,H,D,R,T", [(1, 64, 64, 2, 16), (33, 100, 128, 2, 30), (70, 256, 256, 1, 32), (4200, 200, 256, 1, 32),
                                       (31, 512, 512, 2, 100), (2300, 500, 512, 2, 128), (17, 768, 1024, 1, 128), (4100, 1024, 1024, 1, 128)])
@pytest.mark.parametrize("with_ln", [True, False])
def test_what_the_training_form_keeps(B, H, D, R, T, with_ln):
    """Codes and scores of the form without gradients, bit for bit; z, the stages' inputs and the rows' statistics against 64 bits."""
    gen = torch.Generator(device=DEV).manual_seed(B + D + 1)
    J, NB = 4, D // 64
    x, w = 1.5 * _randn(gen, B, H) + 0.3, _randn(gen, R, J, NB, 64, 64) / math.sqrt(64 * D)
    lw, lb = (1 + 0.1 * _randn(gen, H), 0.1 * _randn(gen, H)) if with_ln else (None, None)
    bias = 0.05 * _randn(gen, T * 8) if with_ln else None
    split = ops.bh4_fold_split(w, False)
    codes, scores = ops.bh4_block_front(x, lw, lb, 1e-5, split, R, J, D, bias, T, 0.7, 0.3)
    got = ops.bh4_block_front_train(x, lw, lb, 1e-5, split, R, J, D, bias, T, 0.7, 0.3)
    assert torch.equal(got[0], codes) and torch.equal(got[1], scores)
    _, _, z, stages, stats = got
    few = min(B, 20)
    part = ops.bh4_block_front_train(x[:few], lw, lb, 1e-5, split, R, J, D, bias, T, 0.7, 0.3)
    assert torch.equal(part[2], z[:few]) and torch.equal(part[3], stages[:, :, :few])
    some = list(range(min(B, 40))) + [B - 1]
    h = x[some].double().cpu()
    if with_ln:
        assert _rel(stats[some, 0], h.mean(1)) <= REL and _rel(stats[some, 1], (h.var(1, unbiased=False) + 1e-5).rsqrt()) <= REL
        h = torch.nn.functional.layer_norm(h, (H,), lw.double().cpu(), lb.double().cpu(), 1e-5)
    h = torch.cat([h, torch.zeros(len(some), D - H, dtype=torch.float64)], 1)
    w64, HD, want = w.double().cpu(), _hadamard(D), []
    for r in range(R):
        u = h
        for j in range(J):
            if j > 0:
                assert _rel(stages[r, j - 1][some], u) <= 2 * REL          # (LayerNorm's rounding as large again)
            u = _blocks(w64[r, j], u) @ HD
        want.append(0.7 * u + 0.3 * h)
    assert _rel(z[some], torch.cat(want, 1)[:, :T * 8] + (bias.double().cpu() if with_ln else 0)) <= 2 * REL
    assert torch.equal((z.view(B, T, 8) > 0).mul(2 ** torch.arange(7, -1, -1, device=DEV)).sum(-1).int(), codes)


@pytest.mark.parametrize("B", [40, 9000])
def test_scales_and_rows_of_their_own(B):
    """Any size of gradients and weights, rows of very different sizes side by side, and a row that is not finite stays alone."""
    gen = torch.Generator(device=DEV).manual_seed(B)
    D, J, T = 256, 4, 32
    g, w = _randn(gen, B, D), _randn(gen, 1, J, D // 64, 64, 64) / math.sqrt(64 * D)
    back = lambda g, w: ops.bh4_block_bwd_split(g, ops.bh4_fold_split(w, True), 1, J, D, D, 1.0, 0.0)[0][0]
    want, HD = g[:40].double().cpu(), _hadamard(D)
    for j in range(J - 1, -1, -1):
        want = _blocks(w[0, j].double().cpu().transpose(-1, -2), want @ HD)
    for sg, sw in ((1e20, 1e-6), (1e-25, 1e6), (1e-8, 1e-4), (1e-3, 1e8)):
        assert _rel(back(g * sg, w * sw)[:40].double() / (sg * sw ** 4), want) <= REL
    base = back(g, w)
    y = g.clone()
    y[3] *= 1e-15
    y[5] *= 1e15
    y[7] = 0
    y[11, 3], y[12, 9] = float("nan"), float("inf")
    got = back(y, w)
    rows = [i for i in range(40) if i not in (3, 5, 7, 11, 12)]
    assert torch.equal(got[rows], base[rows])
    assert _rel(got[3].double() * 1e15, want[3]) <= REL and _rel(got[5].double() * 1e-15, want[5]) <= REL
    assert torch.equal(got[7], torch.zeros_like(got[7])) and got[11].isnan().all() and got[12].isnan().all()
    # the forward: a power of two changes no code
    front = lambda x: ops.bh4_block_front(x, None, None, 0.0, ops.bh4_fold_split(w, False), 1, J, D, None, T, 1.0, 0.0)[0]
    codes = front(g)
    for s in (2.0 ** 60, 2.0 ** -60):
        assert torch.equal(front(g * s), codes)
    got = front(y)
    assert torch.equal(got[rows + [7]], torch.cat([codes[rows], torch.zeros_like(codes[:1])]))
    assert not got[11].any() and not got[12].any()                  # NaN is not above zero


# one stage of the backward, few and many workgroups: columns of the weights of very different sizes side by side, each by its own scale
@pytest.mark.parametrize("B,D", [(40, 64), (33, 256), (9000, 256), (70, 512), (50, 1024)])
def test_columns_of_many_sizes(B, D):
    gen = torch.Generator(device=DEV).manual_seed(B + D)
    sizes = 10.0 ** -(torch.arange(64, device=DEV) * 5 % 13)
    g, w = _randn(gen, B, D), _randn(gen, 1, 1, D // 64, 64, 64) / 64 * sizes
    some = list(range(min(B, 40)))
    got = ops.bh4_block_bwd_split(g, ops.bh4_fold_split(w, True), 1, 1, D, D, 1.0, 0.0)[0][0][some].double().cpu()
    want = _blocks(w[0, 0].double().cpu().transpose(-1, -2), g[some].double().cpu() @ _hadamard(D))
    error, size = (t.view(len(some), D // 64, 64).norm(dim=(0, 1)) for t in (got - want, want))
    assert (error / size).max() <= REL


# the same with blocks of different sizes, whose columns have nothing to do with each other
@pytest.mark.parametrize("B,D", [(33, 128), (33, 256), (9000, 256), (70, 512), (50, 1024), (4100, 1024)])
def test_blocks_of_many_sizes(B, D):
    gen = torch.Generator(device=DEV).manual_seed(B + D)
    sizes = (10.0 ** -(torch.arange(64, device=DEV) * 5 % 13)).view(1, 1, 64) * (10.0 ** -(torch.arange(D // 64, device=DEV) * 5 % 9)).view(-1, 1, 1)
    g, w = _randn(gen, B, D), _randn(gen, 1, 1, D // 64, 64, 64) / 64 * sizes
    some = list(range(min(B, 40)))
    got = ops.bh4_block_bwd_split(g, ops.bh4_fold_split(w, True), 1, 1, D, D, 1.0, 0.0)[0][0][some].double().cpu()
    want = _blocks(w[0, 0].double().cpu().transpose(-1, -2), g[some].double().cpu() @ _hadamard(D))
    assert ((got - want).norm(dim=0) / want.norm(dim=0)).max() <= REL


# Two stages of the forward, few and many workgroups, where the size of a result comes from a small column of the weights and a large
# input as much as from a large column and a small input ("few": within what is scaled together); nor do inputs count that nothing is
# multiplied with.  The error is what it is on numbers of one size, and no larger than that of the kernel with fp32 products (beside
# "zeros", where a third of that one's additions are of zeros and round nothing, while a product is split as ever).
@pytest.mark.parametrize("B,D", [(40, 64), (33, 128), (33, 256), (9000, 256), (70, 512), (2300, 512), (50, 1024), (4100, 1024)])
@pytest.mark.parametrize("kind", ["few", "columns", "blocks", "norm", "zeros"])
def test_columns_against_their_inputs(B, D, kind):
    gen = torch.Generator(device=DEV).manual_seed(B + D)
    J, NB, T = 2, D // 64, D // 8
    x, w = _randn(gen, B, D), _randn(gen, 1, J, NB, 64, 64) / math.sqrt(64 * D)
    lw = lb = None
    decades = 1.5 if kind == "few" else 12
    spread = lambda *shape: 10.0 ** (decades * torch.rand(*shape, generator=gen, device=DEV) - decades / 2)
    w[0, 1] *= spread(NB, 1, 64)                                    # (the second stage's meet numbers of one size)
    if kind == "zeros":
        w[0, 0, :, :, ::3] = 0
        x[:, ::3] *= 1e12
    else:
        e = spread(NB, 1, 1 if kind == "blocks" else 64).expand(NB, 1, 64)
        w[0, 0] *= e
        if kind == "norm":
            lw, lb = (1 + 0.1 * _randn(gen, D)) / e.reshape(D), 0.1 * _randn(gen, D) / e.reshape(D)
        else:
            x /= e.reshape(D)
    some = list(range(min(B, 40))) + [B - 1]
    u = x[some].double().cpu()
    if lw is not None:
        u = torch.nn.functional.layer_norm(u, (D,), lw.double().cpu(), lb.double().cpu(), 1e-5)
    first = _blocks(w[0, 0].double().cpu(), u) @ _hadamard(D)
    want = _blocks(w[0, 1].double().cpu(), first) @ _hadamard(D)
    _, _, z, stages, _ = ops.bh4_block_front_train(x, lw, lb, 1e-5, ops.bh4_fold_split(w, False), 1, J, D, None, T, 1.0, 0.0)
    folded = ops.bh4_fold_mode(w, 0)
    plain = (ops.bh4_block_hash_train(x, folded, None, T, 1.0, 0.0) if lw is None else
             ops.ln_bh4_block_hash_train(x, lw, lb, 1e-5, folded, None, T, 1.0, 0.0))
    limit = lambda t, want: REL if kind == "zeros" else min(REL, _rel(t, want))
    assert _rel(stages[0, 0][some], first) <= limit(plain[3][0, 0][some], first)
    assert _rel(z[some], want) <= limit(plain[2][some], want)
    # without gradients the same codes, whichever form of the kernel and whatever the neighbours
    few = min(B, 20)
    codes, scores = ops.bh4_block_front(x[:few], lw, lb, 1e-5, ops.bh4_fold_split(w, False), 1, J, D, None, T, 1.0, 0.0)
    got = ops.bh4_block_front_train(x, lw, lb, 1e-5, ops.bh4_fold_split(w, False), 1, J, D, None, T, 1.0, 0.0)
    assert torch.equal(codes, got[0][:few]) and torch.equal(scores, got[1][:few])


# the repeats take turns at groups of 128 tiles of 16 tokens: the last group whole, a tile short or a tile over
@pytest.mark.parametrize("B,D,R", [(2048, 512, 2), (2049, 256, 3), (4080, 512, 2), (4112, 64, 4)])
def test_every_tile_of_every_repeat(B, D, R):
    gen = torch.Generator(device=DEV).manual_seed(B)
    J, T = 4, R * D // 8
    x, w = _randn(gen, B, D), _randn(gen, R, J, D // 64, 64, 64) / math.sqrt(64 * D)
    split = ops.bh4_fold_split(w, False)
    front = lambda rows: ops.bh4_block_front(rows, None, None, 1e-5, split, R, J, D, None, T, 0.7, 0.3)
    whole, parts = front(x), [front(x[i:i + 200]) for i in range(0, B, 200)]
    for k in range(2):
        assert torch.equal(whole[k], torch.cat([p[k] for p in parts]))
