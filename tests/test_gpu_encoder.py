"""The encoder's products and attention on the fp16 matrix cores (csrc/linear.hip, csrc/attention.hip) against 64 bits, and the rule
that takes a call to them."""
from argparse import Namespace

import pytest
import torch

import lookupffn_amd
from lookupffn_amd import encoder, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _randn(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed + sum(shape)), device=DEV)


def _rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


# A product of two split numbers is off by at most 2^-22 of itself, a running sum by 2^-24 of itself in each of 3 K / 16 instructions
# (of either sign: their root counts): K = 1024, 2^-22 + 14 * 2^-24 = 1.1e-6 at worst; a quarter of that is what rounding leaves.
LINEAR_REL = 5e-7


# sizes around the tiles of the three forms (64 x 64, 128 x 128, 128 x 256) and one size that gets each of the larger two
@pytest.mark.parametrize("M,N,K,sets", [(1, 64, 32, 1), (63, 65, 64, 3), (64, 128, 512, 2), (129, 200, 96, 3), (700, 512, 512, 3),
                                        (8192, 512, 512, 1), (16333, 768, 768, 3), (4097, 1024, 1024, 1)])
def test_linear_against_64_bits(M, N, K, sets):
    x, w, b = _randn(M, K), [_randn(N, K, seed=s) / K ** 0.5 for s in range(sets)], [_randn(N, seed=9 + s) for s in range(sets)]
    res = _randn(M, N, seed=3)
    got = ops.linear(x, w, [b[0], None, b[-1]][:sets], res)
    rows = torch.randperm(M)[:512].tolist() + [0, M - 1]
    for s in range(sets):
        want = x[rows].double().cpu() @ w[s].double().cpu().T + res[rows].double().cpu()
        if s != 1:
            want += [b[0], None, b[-1]][s].double().cpu()
        assert _rel(got[s][rows], want) <= LINEAR_REL
    assert torch.equal(got, ops.linear(x, w, [b[0], None, b[-1]][:sets], res))


@pytest.mark.parametrize("M", [50, 5000])
def test_linear_keeps_scales_and_infinities(M):
    N = K = 256
    x, w = _randn(M, K), _randn(N, K, seed=1)
    for sx, sw in ((1e-20, 1e15), (1e6, 1e8), (1e-8, 1e-12)):
        got = ops.linear(x * sx, [w * sw], [None], None)[0]
        assert _rel(got, (x * sx).double().cpu() @ (w * sw).double().cpu().T) <= LINEAR_REL
    x[3, 5], x[7, 9], x[9, 1] = float("inf"), -float("inf"), float("nan")
    x[11] = 1e-3
    x[11, 40] = 3e38                        # a row that outgrows its beginning
    x[12, :32] = 0
    w[5, 9] = 0                             # 0 * inf
    want = torch.nn.functional.linear(x.cpu(), w.cpu())
    got = ops.linear(x, [w], [None], None)[0].cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
    assert torch.equal(got.isneginf(), want.isneginf())
    keep = [m for m in range(M) if m not in (3, 7, 9)]
    exact = x[keep].double().cpu() @ w.double().cpu().T
    finite = want[keep].isfinite()
    assert (((got[keep].double() - exact).abs() / exact.norm(dim=1, keepdim=True))[finite]).max() <= 1e-6


# Both ways to the products (with LayerNorm's rows split beforehand only where there are rows enough to ask for it) against 64 bits where
# some columns of x are far larger than others and meet weights of zero: what is left is as exact as if they were not there.  Rows that
# are larger where their scale's sample does not see it, samples of zeros, and numbers near either end of fp32.
@pytest.mark.parametrize("M,K", [(40, 64), (130, 768), (5000, 512)])
@pytest.mark.parametrize("large", [1e4, 1e6, 1e9, 1e30])
@pytest.mark.parametrize("where", ["first", "last", "unseen", "seen"])
def test_linear_of_rows_of_many_sizes(M, K, large, where):
    N = 200
    x, w = _randn(M, K), _randn(N, K, seed=1) / K ** 0.5
    seen = torch.zeros(K, dtype=torch.bool, device=DEV)             # (a fourth of the row begins with its share of the sample)
    for c in range(4):
        seen[c * K // 4:c * K // 4 + 8] = True
    part = {"first": slice(0, 32), "last": slice(K - 32, K), "unseen": ~seen, "seen": seen}[where]
    for rows in (x, w):                     # every third row; the others are what they were
        big, other = rows.clone(), (w if rows is x else x).clone()
        big[::3, part] *= large
        other[:, part] = 0
        # (unseen: the large numbers' products are zero and the sample's are left)
        a, b = (big, other) if rows is x else (other, big)
        got, want = ops.linear(a, [b], [None], None)[0], a.double().cpu() @ b.double().cpu().T
        # 2^-44 of a row's largest number is lost of each at most: beyond 2^21 of the rest, that bound takes the products' place
        share = LINEAR_REL + (0 if large <= 1e6 else 2.0 ** -44 * large * 2)
        if share < 1:
            assert _rel(got, want) <= share
    norm, other = torch.ones(K, device=DEV), w.clone()
    norm[part], other[:, part] = large, 0
    got = ops.linear_norm(x, norm, None, 1e-5, [other], [None])[0]
    want = torch.nn.functional.layer_norm(x.double().cpu(), (K,), norm.double().cpu(), None, 1e-5) @ other.double().cpu().T
    assert share >= 1 or _rel(got, want) <= share + 2.0 ** -22
    sample = x.clone()
    sample[:, seen] = 0                     # nothing to be seen of the row
    for size in (1.0, 1e-10, 1e-25, 1e12, 1e30):
        got = ops.linear(sample * size, [w], [None], None)[0]
        assert _rel(got, (sample * size).double().cpu() @ w.double().cpu().T) <= LINEAR_REL
    for sx, sw in ((1e-37, 1e20), (1e37, 1e-20), (1e-30, 1e-5), (3e37, 1e-30)):
        got = ops.linear(x * sx, [w * sw], [None], None)[0]
        assert _rel(got, (x * sx).double().cpu() @ (w * sw).double().cpu().T) <= LINEAR_REL
    assert torch.equal(ops.linear(torch.zeros_like(x), [w], [None], None)[0], torch.zeros(M, N, device=DEV))


# tiles of 128 x 192: whole rounds and a remainder of rows, a last tile of 124 and of one column, one and three matrices, one step of k
@pytest.mark.parametrize("M,N,K,sets", [(6145, 768, 768, 1), (6145, 700, 32, 1), (6700, 577, 96, 1), (2103, 768, 64, 3)])
def test_linear_in_tiles_of_192_columns(M, N, K, sets):
    x, w, b = _randn(M, K), [_randn(N, K, seed=s) / K ** 0.5 for s in range(sets)], [_randn(N, seed=9 + s) for s in range(sets)]
    w[-1][N - 1] *= 1e9                     # the rows of half a piece have scales of their own
    x[M - 1, K - 1] = float("inf")
    got = ops.linear(x, w, b, None)
    for s in range(sets):
        want = x.double().cpu() @ w[s].double().cpu().T + b[s].double().cpu()
        assert _rel(got[s][:-1, :-1], want[:-1, :-1]) <= LINEAR_REL and _rel(got[s][:-1, -1], want[:-1, -1]) <= LINEAR_REL
        assert torch.equal(got[s][-1].double().cpu(), want[-1])
    assert torch.equal(got, ops.linear(x, w, b, None))


# rows and columns around the tiles of 128, 192 and 256 columns (the last three: one size that gets each), K around the 256 numbers of a
# wavefront's load, LayerNorm with and without weights
@pytest.mark.parametrize("M,N,K,sets", [(1, 1, 32, 1), (129, 200, 288, 3), (300, 64, 2048, 2), (300, 130, 1056, 1), (127, 577, 736, 3),
                                        (4000, 768, 768, 3), (8192, 512, 512, 1), (16333, 512, 512, 3)])
def test_linear_of_a_norm(M, N, K, sets):
    x, w, b = 3 * _randn(M, K) + 1, [_randn(N, K, seed=s) / K ** 0.5 for s in range(sets)], [_randn(N, seed=9 + s) for s in range(sets)]
    x[M // 2] *= 1e6
    w[-1][N - 1] *= 1e9                     # rows have scales of their own
    nw, nb = (None, None) if M == 300 else (1 + 0.1 * _randn(K, seed=5), _randn(K, seed=6))
    bias = [b[0], None, b[-1]][:sets]
    got = ops.linear_norm(x, nw, nb, 1e-5, w, bias)
    rows = sorted(set(torch.randperm(M)[:512].tolist() + [0, M // 2, M - 1]))
    h = torch.nn.functional.layer_norm(x[rows].double().cpu(), (K,), *(t if t is None else t.double().cpu() for t in (nw, nb)), 1e-5)
    for s in range(sets):
        want = h @ w[s].double().cpu().T + (0 if bias[s] is None else bias[s].double().cpu())
        # the norm's mean and variance are sums of K / 64 + 6 additions of 2^-24, either sign: 2^-22 beside the products' bound
        last = [N - 1]
        assert _rel(got[s][rows][:, last], want[:, last]) <= LINEAR_REL + 2.0 ** -22
        assert N == 1 or _rel(got[s][rows][:, :-1], want[:, :-1]) <= LINEAR_REL + 2.0 ** -22
    assert torch.equal(got, ops.linear_norm(x, nw, nb, 1e-5, w, bias))


@pytest.mark.parametrize("M", [130, 4000])
def test_linear_of_a_norm_keeps_infinities(M):
    N = K = 768
    x, w, nw, nb = _randn(M, K), _randn(N, K, seed=1), 1 + 0.1 * _randn(K, seed=5), _randn(K, seed=6)
    x[3, 5], x[9, 1] = float("inf"), float("nan")
    x[20] = 0                               # no variance
    w[5, 9], w[7, 11] = float("inf"), float("nan")
    w[8, :700] = 1e-30
    want = torch.nn.functional.linear(torch.nn.functional.layer_norm(x, (K,), nw, nb), w).cpu()
    got = ops.linear_norm(x, nw, nb, 1e-5, [w], [None])[0].cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
    assert torch.equal(got.isneginf(), want.isneginf())
    finite = want.isfinite()
    h = torch.nn.functional.layer_norm(x.double().cpu(), (K,), nw.double().cpu(), nb.double().cpu())
    # of |h| |w|: 2^-22 for the split and for the norm, 2^-24 in each of 3 K / 16 instructions, either sign: 12 * 2^-24
    bound = h.norm(dim=1, keepdim=True) * w.double().cpu().norm(dim=1) * (2 * 2.0 ** -22 + 12 * 2.0 ** -24)
    assert ((got.double() - h @ w.double().cpu().T).abs() <= bound)[finite].all()
    # infinities in the norm's own weights reach every product of their column
    nw[40] = float("inf")
    want = torch.nn.functional.linear(torch.nn.functional.layer_norm(x, (K,), nw, nb), w).cpu()
    got = ops.linear_norm(x, nw, nb, 1e-5, [w], [None])[0].cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
    assert torch.equal(got.isneginf(), want.isneginf())
    # equal numbers whose square fp32 does not hold: their variance is none (the library's is inf - inf)
    x[:], nw[40] = 1e30, 1
    got = ops.linear_norm(x, nw, nb, 1e-5, [w[9:]], [None])[0]
    assert _rel(got, (nb.double().cpu() @ w[9:].double().cpu().T).expand(M, -1)) <= LINEAR_REL


def _exact_attention(q, k, v, mask):
    q, k, v = (t.double().cpu().permute(0, 2, 1, 3) for t in (q, k, v))
    bias = -1000 * (1 - mask.double().cpu()[:, None, None])
    return (torch.softmax(q @ k.transpose(-1, -2).contiguous() / 8 + bias, -1) @ v).permute(0, 2, 1, 3)


# lengths around the 64 keys of a step and the 128 queries of a workgroup, and the longest
@pytest.mark.parametrize("B,L,heads", [(1, 1, 1), (2, 33, 3), (3, 64, 8), (2, 65, 12), (1, 127, 2), (2, 129, 5), (4, 512, 12), (1, 2048, 2)])
def test_attention_against_64_bits(B, L, heads):
    q, k, v = (_randn(B, L, heads, 64, seed=s) for s in range(3))
    mask = (torch.arange(L, device=DEV)[None] < torch.randint((L + 1) // 2, L + 1, (B, 1), device=DEV)).float()
    got = ops.attention(q, k, v, mask)
    # scores up to 8 are off by 2^-22 of |q| |k| / 8, weights and results by as much again: 8 * 2^-22 at worst
    assert _rel(got, _exact_attention(q, k, v, mask)) <= 1e-6
    assert torch.equal(got, ops.attention(q, k, v, mask))


def test_attention_masks_scales_and_infinities():
    B, L, heads = 6, 150, 4
    q, k, v = (_randn(B, L, heads, 64, seed=s) for s in range(3))
    mask = torch.ones(B, L, device=DEV)
    mask[1] = 0                                                     # nothing but padding
    mask[2] = -float("inf")                                         # masks of another convention
    mask[3, 50:] = torch.finfo(torch.float32).min
    mask[4] = torch.rand(L, device=DEV)
    q[5], k[5], v[5] = q[5] * 1e12, k[5] * 1e-12, v[5] * 1e-20
    got, want = ops.attention(q, k, v, mask), _exact_attention(q, k, v, mask)
    for b in (0, 1, 3, 4, 5):
        assert _rel(got[b], want[b]) <= 1e-6, b
    assert torch.equal(got[2], torch.zeros_like(got[2]))            # as torch's attention has it
    q[0, 3, 1, 5], k[1, 70, 2, 3], v[3, 8, 1] = float("inf"), float("inf"), float("nan")
    k[4, 140], v[4, 141] = k[4, 140] * 1e6, v[4, 141] * 1e6         # keys and values that outgrow the first ones
    got, want = ops.attention(q, k, v, mask), _exact_attention(q, k, v, mask)
    for b in (0, 1, 3, 4, 5):
        assert torch.equal(got[b].isnan().cpu(), want[b].isnan()), b
        assert _rel(got[b].nan_to_num(), want[b].nan_to_num()) <= 2e-6, b


# Steps of 64 keys: values that grow from one to the next in all or some columns, columns and keys of many sizes, first keys that say
# nothing of the others.
@pytest.mark.parametrize("L", [70, 200, 512])
@pytest.mark.parametrize("columns", [1, 3, 64])
def test_attention_of_many_sizes(L, columns):
    B, heads = 2, 3
    q, k, v = (_randn(B, L, heads, 64, seed=s) for s in range(3))
    mask = torch.ones(B, L, device=DEV)

    def close(q, k, v, share=1e-6):                     # column for column
        got, want = ops.attention(q, k, v, mask).double().cpu().flatten(0, 2), _exact_attention(q, k, v, mask).flatten(0, 2)
        assert ((got - want).norm(dim=0) / want.norm(dim=0)).max() <= share

    every = 64 // columns
    for f in (1e2, 1e5, 1e12, 1e30):
        grown = v.clone()
        grown[:, 65::9, :, ::every] *= f                # (of one in nine keys behind the first step's)
        grown[:, 65::30, :, ::every] *= f if f < 1e30 else 1e6
        close(q, k, grown)
        small = v.clone()
        small[:, :65, :, ::every] /= f
        close(q, k, small)
    sizes = v * 10.0 ** (torch.arange(64, device=DEV) % 13 - 6)
    close(q, k, sizes)
    close(q, k * torch.where(torch.arange(L, device=DEV) % 3 == 1, 1e-7, 1.0)[:, None, None], sizes)
    late = v * 1e-20
    late[:, :64] = 0
    close(q, k, late)
    # a value a million times the others' that no query looks at: its column's others are held to 2^-39 of it (values beyond its step
    # are, too): 2^-39 4e6 is 7e-6 at most of a value, a third of that on average of either sign, over at least 70 keys
    k[:, 65], v[:, 65, :, ::every], mask[:, 65] = 0, 1e6, 0
    close(q, k, v, 3e-6)


def _config(hidden, heads):
    return Namespace(hidden_size=hidden, num_attention_heads=heads, attention_head_size=hidden // heads, attention_probs_dropout_prob=0.1,
                     hidden_dropout_prob=0.1, layer_norm_eps=1e-5, ffn_num_table=32, ffn_table_size=256, projection_type="bh4", block_size=1)


@pytest.fixture
def layer():
    torch.manual_seed(3)
    return lookupffn_amd.EncoderLayer(_config(256, 4)).eval().to(DEV)


def _by_library(layer, x, mask):
    att = layer.attention
    return layer.dropout(att._attend(att.LayerNorm(x), mask)) + x


# another norm is called, the layer's own is not; either way the layer is what the library's products give
@pytest.mark.parametrize("form", ["own", "hook", "subclass", "class method", "no weights", "too few rows"])
def test_the_norm_in_the_products(layer, form, monkeypatch):
    att = layer.attention
    torch.nn.init.normal_(att.LayerNorm.weight, 1, 0.1)
    rows = 40 if form == "too few rows" else 600
    x, mask = _randn(4, rows, 256), torch.ones(4, rows, device=DEV)
    norms, calls = [], []
    if form == "hook":
        att.LayerNorm.register_forward_hook(lambda *a: norms.append(1))
    if form == "subclass":
        forward = lambda self, h: norms.append(1) or 2 * torch.nn.LayerNorm.forward(self, h)
        att.LayerNorm = type("Norm", (torch.nn.LayerNorm,), {"forward": forward})(256).to(DEV)
    if form == "class method":
        norm_forward = torch.nn.LayerNorm.forward
        monkeypatch.setattr(torch.nn.LayerNorm, "forward", lambda self, h: norms.append(1) or norm_forward(self, h))
    if form == "no weights":
        att.LayerNorm = torch.nn.LayerNorm(256, eps=1e-3, elementwise_affine=False)
    monkeypatch.setattr(encoder.ops, "linear_norm", lambda *a: calls.append(1) or torch.ops.lookupffn.linear_norm(*a))
    with torch.no_grad():
        got = att(x, mask)
        assert bool(calls) == (form in ("own", "no weights")) and bool(norms) == (form in ("hook", "subclass", "class method"))
        want = att._attend(att.LayerNorm(x), mask)
    assert _rel(got, want.double().cpu()) <= 1e-6


@pytest.mark.parametrize("form", ["plain", "strided", "bool mask", "half mask", "strided mask", "no bias", "one token"])
def test_the_kernels_agree_with_the_library_path(layer, form, monkeypatch):
    x, mask = _randn(3, 77, 256), (torch.arange(77, device=DEV)[None] < torch.tensor([[77], [50], [39]], device=DEV)).float()
    if form == "strided":
        x = _randn(3, 256, 77).transpose(1, 2)
    if form == "bool mask":
        mask = mask.bool().float().to(torch.int64)
    if form == "half mask":
        mask = mask.half()
    if form == "strided mask":
        mask = mask.t().contiguous().t()
    if form == "no bias":
        layer.attention.key.bias = None
    if form == "one token":
        x, mask = x[:1, :1], mask[:1, :1]
    calls = []
    monkeypatch.setattr(encoder.ops, "attention", lambda *a: calls.append(1) or torch.ops.lookupffn.attention(*a))
    with torch.no_grad():
        got = layer._attention_and_residual(x, mask)
        assert calls
        assert torch.equal(got, layer.attention(x, mask) + x)
        want = _by_library(layer, x, mask)
    assert got.shape == want.shape and got.is_contiguous()
    assert _rel(got, want.double().cpu()) <= 1e-6


@pytest.mark.parametrize("form", ["hook", "pre-hook", "global hook", "other linear", "own forward", "own attention", "own attend", "subclass",
                                  "Attention.attention", "Attention.transpose_for_scores", "Attention._attend", "Attention.forward",
                                  "Linear.forward", "Dropout.forward", "gradient", "autocast",
                                  "dropout", "train", "double", "heads", "wide mask", "vmap", "tangent", "misaligned"])
def test_other_calls_keep_the_library_path(layer, form, monkeypatch):
    calls, seen = [], []
    monkeypatch.setattr(encoder.ops, "attention", lambda *a: calls.append(1) or torch.ops.lookupffn.attention(*a))
    x, mask = _randn(2, 40, 256), torch.ones(2, 40, device=DEV)
    att = layer.attention
    run = lambda: att(x, mask)
    grad, handle = torch.no_grad(), None
    if form == "hook":
        att.query.register_forward_hook(lambda *a: seen.append(1))
    if form == "pre-hook":
        att.dense.register_forward_pre_hook(lambda *a: seen.append(1))
    if form == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(1))
    if form == "other linear":
        class Twice(torch.nn.Linear):
            def forward(self, t):
                seen.append(1)
                return 2 * super().forward(t)
        att.value.__class__ = Twice
    if form == "own forward":
        inner = att.value.forward
        att.value.forward = lambda t: seen.append(1) or inner(t)
    if form == "own attention":
        inner_attention = att.attention
        att.attention = lambda *a: seen.append(1) or inner_attention(*a)
    if form == "own attend":
        inner_attend = att._attend
        att._attend = lambda *a: seen.append(1) or inner_attend(*a)
    if "." in form:                         # a class that has been given another method
        kind, name = form.split(".")
        kind = {"Attention": encoder.Attention, "Linear": torch.nn.Linear, "Dropout": torch.nn.Dropout}[kind]
        inner_method = getattr(kind, name)
        monkeypatch.setattr(kind, name, lambda *a: seen.append(1) or inner_method(*a))
        run = lambda: layer._attention_and_residual(x, mask)
    if form == "subclass":
        class Other(encoder.Attention):
            def attention(self, *a):
                seen.append(1)
                return super().attention(*a)
        att.__class__ = Other
    if form == "gradient":
        grad = torch.enable_grad()
    if form == "autocast":
        grad = torch.autocast("cuda", torch.float16)
        layer.requires_grad_(False)
    if form == "dropout":
        layer.train()
    if form == "train":                     # (as with gradients)
        layer.train()
        layer.dropout.p = layer.attention.dropout.p = 0.0
        run = lambda: layer._attention_and_residual(x, mask)
    if form == "double":
        att.double()
        x = x.double()
    if form == "heads":
        att.num_attention_heads, att.attention_head_size = 8, 32
    if form == "wide mask":
        mask = torch.ones(1, 40, device=DEV)
    if form == "vmap":
        layer.requires_grad_(False)
        run = lambda: torch.vmap(lambda t: att(t[None], mask[:1])[0])(x)
    if form == "tangent":
        def run():
            with torch.autograd.forward_ad.dual_level():
                t = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
                with torch.no_grad(), torch.nn.attention.sdpa_kernel(torch.nn.attention.SDPBackend.MATH):
                    assert att(t, mask) is not None
        grad = torch.enable_grad()
        layer.requires_grad_(False)
    if form == "misaligned":
        flat = torch.empty(256 * 256 + 1, device=DEV)
        att.key.weight.data = flat[1:].view(256, 256).copy_(att.key.weight.data)
        assert att.key.weight.data_ptr() % 16 != 0
    try:
        with grad:
            run()
    finally:
        if handle is not None:
            handle.remove()
    assert not calls or form in ("Attention.forward", "Dropout.forward")         # (called, and goes on to the kernels)
    assert seen or form in ("gradient", "autocast", "dropout", "train", "double", "heads", "wide mask", "vmap", "tangent", "misaligned")


def test_encoder_layer_in_a_graph(layer):
    x, mask = _randn(2, 70, 256), torch.ones(2, 70, device=DEV)
    with torch.no_grad():
        for _ in range(3):
            layer(x, mask)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, mask)
        for seed in range(3):
            x.copy_(_randn(2, 70, 256, seed=seed))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, layer(x, mask))
