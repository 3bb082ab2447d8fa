"""weighted_gather_add and its backward on flat row numbers at the sizes where the choice of kernels, the row lists or the
tiles can go wrong, against float64 sums of the same values.

Bounds: an fp32 sum of n products is within n * 2^-24 of the sum of their magnitudes; the comparisons below use that sum
itself (the operator on absolute values in float64) as the scale of every element."""
import ctypes

import numpy as np
import pytest
import torch

import lookupffn_amd
from lookupffn_amd import _lib, ops
from tests import _cabi as cabi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(B, I, rows, Dv, form, dtype=torch.float32, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + B + I + Dv)
    if form == "tables":
        idx = torch.randint(0, 256, (B, I), generator=g, device=DEV, dtype=torch.int32)
        idx += 256 * torch.arange(I, device=DEV, dtype=torch.int32)[None]
    elif form == "one row":
        idx = torch.full((B, I), rows - 1, device=DEV, dtype=torch.int32)
    else:
        idx = torch.randint(0, rows, (B, I), generator=g, device=DEV, dtype=torch.int32)
    if form == "tables but one":
        idx = torch.randint(0, 256, (B, I), generator=g, device=DEV, dtype=torch.int32)
        idx += 256 * torch.arange(I, device=DEV, dtype=torch.int32)[None]
        idx[B - 1, I - 1] = 3
    src = torch.randn(rows, Dv, generator=g, device=DEV).to(dtype)
    w = torch.randn(B, I, generator=g, device=DEV).to(dtype)
    grad = torch.randn(B, Dv, generator=g, device=DEV).to(dtype)
    return idx, src, w, grad


def _reference(idx, src, w, grad):
    """(out, grad_weights, grad_source) in float64 by columns of the index array."""
    src, w, grad = src.double(), w.double(), grad.double()
    out, gw, gs = torch.zeros_like(grad), torch.empty_like(w), torch.zeros_like(src)
    for i in range(idx.shape[1]):
        rows = idx[:, i].long()
        out += w[:, i, None] * src[rows]
        gw[:, i] = (grad * src[rows]).sum(1)
        gs.index_add_(0, rows, w[:, i, None] * grad)
    return out, gw, gs


def _close(got, want, scale, terms):
    # + 2^-23: the result's own rounding
    assert ((got.double() - want).abs() <= scale * (terms * 2.0 ** -24 + 2.0 ** -23)).all()


SHAPES = [
    # (tokens, columns, rows, Dv): table-major forms with ragged tiles, a table split, the smallest sorted lists, rows that
    # are no multiple of 256, more tokens than one chunk, a single 64-column slice pair
    (4096, 128, 128 * 256, 512), (2103, 64, 64 * 256, 768), (1031, 32, 32 * 256, 1024), (4099, 130, 130 * 256, 64),
    (257, 126, 1000, 192), (100, 8, 77, 8192), (16500, 8, 8 * 256, 128), (1, 6, 24, 1 << 20), (513, 62, 62 * 256, 320),
]


@pytest.mark.parametrize("form", ["tables", "any", "tables but one", "one row"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_weighted_gather_add_and_gradients(shape, form):
    B, I, rows, Dv = shape
    if form.startswith("tables") and rows != 256 * I:
        pytest.skip("not tables of 256 rows")
    idx, src, w, grad = _inputs(B, I, rows, Dv, form)
    src.requires_grad_(), w.requires_grad_()
    out = lookupffn_amd.weighted_gather_add(idx, src, w)
    out.backward(grad)
    want = _reference(idx, src.detach(), w.detach(), grad)
    scale = _reference(idx, src.detach().abs(), w.detach().abs(), grad.abs())
    counts = torch.bincount(idx.reshape(-1), minlength=rows).max().item()
    for got, x, s, terms in zip((out.detach(), w.grad, src.grad), want, scale, (I, Dv, counts)):
        _close(got, x, s, terms)


@pytest.mark.parametrize("shape", [(4096, 128, 128 * 256, 512), (100, 8, 77, 8192), (3000, 62, 62 * 256, 192)], ids=str)
@pytest.mark.parametrize("form", ["tables", "any"])
def test_half_rows_and_gradients(shape, form):
    B, I, rows, Dv = shape
    if form == "tables" and rows != 256 * I:
        pytest.skip("not tables of 256 rows")
    idx, src, w, grad = _inputs(B, I, rows, Dv, form, torch.float16)
    src.requires_grad_(), w.requires_grad_()
    out = lookupffn_amd.weighted_gather_add(idx, src, w)
    out.backward(grad)
    want = _reference(idx, src.detach(), w.detach(), grad)
    scale = _reference(idx, src.detach().abs(), w.detach().abs(), grad.abs())
    counts = torch.bincount(idx.reshape(-1), minlength=rows).max().item()
    for got, x, s, terms in zip((out.detach(), w.grad, src.grad), want, scale, (I, Dv, counts)):
        assert got.dtype == torch.float16
        # fp32 sums, then one rounding to half (2^-11 of the value, 2^-25 below the normal range)
        assert ((got.double() - x).abs() <= s * terms * 2.0 ** -24 + x.abs() * 2.0 ** -10.9 + 2.0 ** -24).all()


def test_scatter_rows_accumulates_and_clamps():
    B, I, rows, Dv = 700, 64, 300, 256
    idx, _, w, grad = _inputs(B, I, rows, Dv, "any")
    idx[3, 5], idx[4, 6] = -7, rows + 1000          # clamped into range, as every operator does
    start = torch.randn(rows, Dv, device=DEV)
    out = start.clone()
    lib = _lib.load()
    ws = ops._workspace(out.device, "lffn_scatter_rows_workspace_bytes", B, I, rows, Dv)
    assert ws is not None
    rc = lib.lffn_scatter_rows(idx.data_ptr(), grad.data_ptr(), w.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, I, rows,
                               Dv, 0, 1, _lib.stream_of(out))
    assert rc == 0
    clamped = idx.clamp(0, rows - 1)
    src = torch.zeros(rows, Dv, device=DEV)
    want = _reference(clamped, src, w, grad)[2] + start.double()
    scale = _reference(clamped, src, w.abs(), grad.abs())[2] + start.abs().double()
    _close(out, want, scale, torch.bincount(clamped.reshape(-1)).max().item() + 1)


# The layer in one launch: column passes of 256 below, at and past their edges and past the four that go together, table
# counts around the eight wavefronts' shares, one to three repeats, more stages than are requested together
@pytest.mark.parametrize("B,H,D,R,J,T,Do", [(1, 256, 256, 1, 4, 1, 64), (3, 250, 256, 2, 5, 63, 260), (5, 512, 512, 1, 1, 64, 512),
                                            (2, 768, 1024, 1, 4, 128, 1284), (9, 1024, 1024, 4, 4, 512, 1024),
                                            (260, 512, 512, 1, 4, 33, 256), (257, 1024, 1024, 4, 4, 480, 1088)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_one_launch_layer_on_rows_of_every_format(B, H, D, R, J, T, Do, dtype):
    gen = torch.Generator().manual_seed(B + H + T)
    rand = lambda *s: torch.randn(*s, generator=gen)
    x, res = rand(B, H), rand(B, Do)
    lw, lb = 1 + 0.1 * rand(H), 0.1 * rand(H)
    diag = torch.sign(rand(R, J, D)) / D ** 0.5
    pbias, obias = 0.01 * rand(T * 8), 0.001 * rand(Do)
    tables = (0.02 * rand(T, 256, Do)).to(dtype)
    code, score, _ = cabi.ln_project_hash(x.numpy(), lw.numpy(), lb.numpy(), 1e-5, diag.numpy(), pbias.numpy(), T)
    rows = tables.double()[torch.arange(T)[None], torch.from_numpy(code).long()]             # [B, T, Do]
    products = rows * torch.from_numpy(score).double()[:, :, None]
    want = products.sum(1) + obias.double() + res.double()
    dev = {k: v.cuda() for k, v in dict(lw=lw, lb=lb, diag=diag, pbias=pbias, tables=tables, obias=obias, x=x, res=res).items()}
    p = lambda k: dev[k].data_ptr()
    block = _lib.FusedLayer(p("lw"), p("lb"), p("diag"), p("pbias"), p("tables"), p("obias"), H, D, R, J, T, 256, Do, 1e-5,
                            float(np.float32(0.7)), float(np.float32(1 - 0.7)))
    out = torch.full((B, Do), float("nan"), device="cuda")
    fmt = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    _lib.check(_lib.load().lffn_lookup_ffn_fused_layer_rows(ctypes.byref(block), fmt, p("x"), p("res"), out.data_ptr(), B,
                                                            torch.cuda.current_stream().cuda_stream), "fused")
    # fp32 sums of T products, exact in the rows: each of T + 8 additions rounds by 2^-24 of a partial sum
    bound = (T + 8) * 2.0 ** -24 * (products.abs().sum(1) + obias.abs() + res.abs())
    assert ((out.cpu().double() - want).abs() <= bound).all()


# The gather by a workgroup per token: both widths of workgroup, table counts around the wavefronts' shares, column passes, table
# sizes other than 256, and the largest batch of it
@pytest.mark.parametrize("B,T,S,Do", [(1, 1, 16, 64), (7, 65, 256, 320), (256, 32, 128, 256), (257, 30, 256, 1088), (512, 512, 256, 64),
                                      (1024, 8, 256, 768)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_gather_of_few_tokens(B, T, S, Do, dtype):
    gen = torch.Generator().manual_seed(B + T)
    code = torch.randint(0, S, (B, T), generator=gen, dtype=torch.int32)
    score = torch.randn(B, T, generator=gen)
    tables = torch.randn(T, S, Do, generator=gen).to(dtype)
    bias, res = torch.randn(Do, generator=gen), torch.randn(B, Do, generator=gen)
    want, scale = bias.double() + res.double(), bias.abs().double() + res.abs().double()
    for t in range(T):
        products = tables[t].double()[code[:, t].long()] * score[:, t].double()[:, None]
        want, scale = want + products, scale + products.abs()
    got = ops.lookup_gather(code.cuda(), score.cuda(), tables.cuda(), bias.cuda(), res.cuda())
    assert ((got.cpu().double() - want).abs() <= (T + 8) * 2.0 ** -24 * scale).all()      # T + 8 additions in fp32


# 64 x 64 blocks: few tokens and many take different forms of the kernel, which do the same additions in the same order
@pytest.mark.parametrize("D,R", [(256, 1), (256, 2), (512, 1), (1024, 1)])
def test_block_kernel_forms_agree(D, R):
    rng = np.random.RandomState(D + R)
    B, few, J, T = 16 * (256 // R) + 5, 37, 3, R * D // 8
    w = (rng.randn(R, J, D // 64, 64, 64) / np.sqrt(64 * D)).astype(np.float32)
    x, bias = rng.randn(B, D - 4).astype(np.float32), (0.05 * rng.randn(T * 8)).astype(np.float32)
    lw, lb = (1 + 0.1 * rng.randn(D - 4)).astype(np.float32), (0.1 * rng.randn(D - 4)).astype(np.float32)
    many = cabi.ln_bh4_block_train(x, lw, lb, 1e-5, w, bias, T)
    for a, b in zip(many, cabi.ln_bh4_block_train(x[:few], lw, lb, 1e-5, w, bias, T)):
        assert np.array_equal(a[:, :, :few] if a.ndim == 4 else a[:few], b)
    assert np.array_equal(cabi.bh4_block(x, w)[0][:few], cabi.bh4_block(x[:few], w)[0])
    g = rng.randn(B, T * 8).astype(np.float32)
    for a, b in zip(cabi.bh4_block_bwd(g, w, D - 4), cabi.bh4_block_bwd(g[:few], w, D - 4)):
        assert np.array_equal(a[..., :few, :], b)


@pytest.mark.parametrize("B", [1, 63, 64, 65, 385, 1100])
def test_block_weight_gradient_over_chunks(B):
    """Chunks of 64 to 512 tokens: sums of B products in fp32, per element within B * 2^-24 of the sum of their magnitudes."""
    rng = np.random.RandomState(B)
    J, D = 2, 128
    sg, x, si = (rng.randn(*s).astype(np.float32) for s in ((J, B, D), (B, D), (1, J - 1, B, D)))
    u = np.stack([x, si[0, 0]]).astype(np.float64).reshape(J, B, D // 64, 64)
    p = sg.astype(np.float64).reshape(J, B, D // 64, 64)
    want, scale = np.einsum("jbno,jbni->jnoi", p, u), np.einsum("jbno,jbni->jnoi", np.abs(p), np.abs(u))
    got = cabi.bh4_block_wgrad(sg, x, si, 1, J)
    assert (np.abs(got - want) <= (B + 4) * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("B", [7200, 14337])
def test_block_weight_gradient_over_long_chunks(B):
    """Chunks of 1024 and 2048 tokens, the last one short; bound as above."""
    torch.manual_seed(B)
    R, J, D = 8, 4, 128
    sg, x, si = (torch.randn(*s, device="cuda") for s in ((R * J, B, D), (B, D), (R, J - 1, B, D)))
    got = lookupffn_amd.ops.bh4_block_wgrad(sg, x, si, R, J)
    for s in range(R * J):
        u = (x if s % J == 0 else si[s // J, s % J - 1]).double().view(B, D // 64, 64).permute(1, 0, 2).contiguous()
        p = sg[s].double().view(B, D // 64, 64).permute(1, 2, 0).contiguous()
        assert ((got[s] - torch.bmm(p, u)).abs() <= (B + 4) * 2.0 ** -24 * torch.bmm(p.abs(), u.abs())).all(), s


# chunks of 2048, 1024 and 512 tokens with a short end, LayerNorm on load in the first stage
@pytest.mark.parametrize("B,D,R", [(31000, 1024, 1), (17000, 512, 2), (4200, 512, 1)])
def test_block_weight_gradient_grows_no_error(B, D, R):
    """Relative error (2-norm) of sums of B products: a sum of n numbers of either sign in a row is rounded n times at n / 2 of its square on
    average, half an ulp at most and a third of that in square.  Runs of 64 products: 32, up to 8 runs 4, four wavefronts 2, up to 17
    chunks 8, a normalised input's own roundings 4."""
    gen = torch.Generator(device="cuda").manual_seed(B)
    J = 2
    sg, x, si = (torch.randn(*s, generator=gen, device="cuda") for s in ((R * J, B, D), (B, D), (R, J - 1, B, D)))
    lw, lb = 1 + 0.1 * torch.randn(D, generator=gen, device="cuda"), 0.1 * torch.randn(D, generator=gen, device="cuda")
    h = torch.nn.functional.layer_norm(x.double(), (D,), lw.double(), lb.double(), 1e-5)
    stats = torch.stack([x.double().mean(1), (x.double().var(1, unbiased=False) + 1e-5).rsqrt()], 1).float().contiguous()
    for got, first in ((lookupffn_amd.ops.ln_bh4_block_wgrad(sg, x, lw, lb, stats, si, R, J), h),
                       (lookupffn_amd.ops.bh4_block_wgrad(sg, x, si, R, J), x)):
        for s in range(R * J):
            u = (first if s % J == 0 else si[s // J, s % J - 1]).double().view(B, D // 64, 64).permute(1, 0, 2).contiguous()
            want = torch.bmm(sg[s].double().view(B, D // 64, 64).permute(1, 2, 0).contiguous(), u)
            assert (got[s].double() - want).norm() <= (50 / 3) ** 0.5 * 2.0 ** -24 * want.norm(), s


# pairs counted in LDS (row numbers of column i in table i) beside pairs that are not, tokens and columns short of a workgroup's 1024 x 4
@pytest.mark.parametrize("B,I,in_tables", [(2047, 9, 1.0), (2048, 13, 1.0), (3000, 12, 0.0), (2049, 33, 0.5), (3073, 70, 0.97)])
def test_row_sums_of_mixed_row_numbers(B, I, in_tables):
    gen = torch.Generator(device="cuda").manual_seed(B)
    rows, Dv = I * 256 - 100, 320
    idx = torch.randint(0, 256, (B, I), generator=gen, device="cuda") + 256 * torch.arange(I, device="cuda")
    other = torch.randint(-300, rows + 300, (B, I), generator=gen, device="cuda")          # (row numbers are held to the range)
    idx = torch.where(torch.rand(B, I, generator=gen, device="cuda") < in_tables, idx, other).int()
    idx[:, 1] = torch.where(torch.arange(B, device="cuda") % 3 == 0, 300, idx[:, 1])      # a row of many pairs
    w, g = torch.randn(B, I, generator=gen, device="cuda"), torch.randn(B, Dv, generator=gen, device="cuda")
    size = ctypes.c_int64()
    assert _lib.load().lffn_scatter_rows_workspace_bytes(B, I, rows, Dv, ctypes.byref(size)) == 0 and size.value > 0
    ws, out = torch.empty(size.value, dtype=torch.uint8, device="cuda"), torch.full((rows, Dv), float("nan"), device="cuda")
    assert _lib.load().lffn_scatter_rows(idx.data_ptr(), g.data_ptr(), w.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, I, rows, Dv,
                                         0, 0, _lib.stream_of(g)) == 0
    at, want, scale = idx.long().clamp(0, rows - 1), torch.zeros(rows, Dv, device="cuda").double(), torch.zeros(rows, Dv, device="cuda").double()
    for i in range(I):
        part = w[:, i:i + 1].double() * g.double()
        want.index_add_(0, at[:, i], part)
        scale.index_add_(0, at[:, i], part.abs())
    most = torch.bincount(at.flatten(), minlength=rows)[:, None]
    assert ((out - want).abs() <= (most + 4) * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("shapes", [[(1, 4)], [(513, 768), (2, 36), (127, 32)], [(2049, 64), (128, 1024), (129, 4), (512, 4096), (3, 8)] + 3 * [(40, 0)]])
def test_sums_of_many_arrays(shapes):
    """At most 17 numbers to a lane, then 3 + 15 additions: 36 roundings of the magnitudes' sum."""
    gen = torch.Generator(device="cuda").manual_seed(len(shapes))
    parts = [torch.randn(s, generator=gen, device="cuda") for s in shapes]
    outs = [torch.full((n,), float("nan"), device="cuda") for _, n in shapes]
    sums = (_lib.Sum * len(shapes))(*[_lib.Sum(p.data_ptr(), o.data_ptr(), n, P) for p, o, (P, n) in zip(parts, outs, shapes)])
    assert _lib.load().lffn_sum_many_f32(sums, len(shapes), _lib.stream_of(parts[0])) == 0
    for p, o in zip(parts, outs):
        assert ((o - p.double().sum(0)).abs() <= 36 * 2.0 ** -24 * p.double().abs().sum(0)).all()


# rows around the copy's 32 and its chunks of 16384; columns that leave threads idle, and more than one workgroup has threads for
@pytest.mark.parametrize("B,Do", [(1, 64), (31, 192), (32, 512), (1000, 1088), (70, 8192), (16384, 64), (16385, 128)])
def test_column_sums_of_the_backwards_copy(B, Do):
    gen = torch.Generator(device="cuda").manual_seed(B)
    T, S, L = 8, 16, _lib.load()
    code = torch.randint(0, S, (B, T), generator=gen, device="cuda", dtype=torch.int32)
    score, g = torch.rand(B, T, generator=gen, device="cuda"), torch.randn(B, Do, generator=gen, device="cuda")
    tables = torch.randn(T, S, Do, generator=gen, device="cuda")
    size = ctypes.c_int64()
    assert L.lffn_lookup_scatter_workspace_bytes(B, T, S, Do, ctypes.byref(size)) == 0
    ws, results = torch.empty(size.value, dtype=torch.uint8, device="cuda"), []
    assert L.lffn_lookup_backward_sums_rows(B, ctypes.byref(size)) == 0
    sums = torch.full((size.value, Do), float("nan"), device="cuda")
    for to in (sums, None):
        gs, gt = torch.empty(B, T, device="cuda"), torch.empty_like(tables)
        assert L.lffn_lookup_backward_sums_f32(code.data_ptr(), score.data_ptr(), g.data_ptr(), tables.data_ptr(), gs.data_ptr(), gt.data_ptr(),
                                               _lib.ptr(to), ws.data_ptr(), ws.numel(), B, T, S, Do, 0, _lib.stream_of(g)) == 0
        results.append((gs, gt))
    assert all(torch.equal(a, b) for a, b in zip(*results))
    got = sums.double().sum(0)                              # each row of it the sum of at most 32 numbers
    assert ((got - g.double().sum(0)).abs() <= 32 * 2.0 ** -24 * g.double().abs().sum(0)).all()


# Both gradients of the layer's gather for few tokens and just past it: row groups of 32 and smaller tables, column passes, every token
# on one row, adding to what is there
@pytest.mark.parametrize("B,T,S,Do", [(1, 1, 256, 64), (5, 9, 16, 320), (64, 3, 32, 1088), (384, 65, 256, 768), (385, 8, 128, 256),
                                      (2048, 3, 256, 64), (2049, 3, 256, 64)])
@pytest.mark.parametrize("skew", [False, True])
def test_gather_gradients_of_few_tokens(B, T, S, Do, skew):
    rng = np.random.RandomState(B + T + S)
    code = np.full((B, T), S - 1, np.int32) if skew else rng.randint(0, S, (B, T)).astype(np.int32)
    score, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    tables, init = rng.randn(T, S, Do).astype(np.float32), rng.randn(T, S, Do).astype(np.float32)
    want, scale = np.zeros((T, S, Do)), np.zeros((T, S, Do))
    for t in range(T):
        products = score[:, t, None].astype(np.float64) * g
        np.add.at(want[t], code[:, t], products)
        np.add.at(scale[t], code[:, t], np.abs(products))
    # products rounded to fp32, summed in fp64, the sum (and the one onto `init`) rounded to fp32
    assert (np.abs(cabi.lookup_scatter(code, score, g, S) - want) <= 2 * 2.0 ** -24 * scale).all()
    got = cabi.lookup_scatter(code, score, g, S, accumulate=True, init=init)
    assert (np.abs(got - want - init) <= 3 * 2.0 ** -24 * (scale + np.abs(init))).all()
    rows = tables[np.arange(T)[None], code].astype(np.float64)                               # [B, T, Do]
    inner = np.einsum("btd,bd->bt", rows, g.astype(np.float64))
    bound = (Do + 8) * 2.0 ** -24 * np.einsum("btd,bd->bt", np.abs(rows), np.abs(g).astype(np.float64))
    assert (np.abs(cabi.lookup_inner(code, g, tables) - inner) <= bound).all()


# Flat row numbers, few tokens: numbers outside the source are clamped, any source size, more columns than go together
@pytest.mark.parametrize("B,I,rows,Dv", [(1, 1, 1, 64), (3, 70, 999, 320), (256, 16, 100, 1088), (385, 9, 4000, 128), (513, 9, 4000, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_operators_on_flat_rows_of_few_tokens(B, I, rows, Dv, dtype):
    gen = torch.Generator().manual_seed(B + I)
    idx = torch.randint(-3, rows + 3, (B, I), generator=gen, dtype=torch.int32)
    src, g, w = (torch.randn(*s, generator=gen).to(dtype) for s in ((rows, Dv), (B, Dv), (B, I)))
    picked = src.double()[idx.long().clamp(0, rows - 1)]                                     # [B, I, Dv]
    want, scale = ((f(picked) * f(w.double())[:, :, None]).sum(1) for f in (lambda t: t, torch.abs))
    got = ops.gather_add(idx.cuda(), src.cuda(), w.float().cuda()).cpu().double()
    assert ((got - want).abs() <= (I + 8) * 2.0 ** -24 * scale).all()
    want, scale = ((f(picked) * f(g.double())[:, None]).sum(2) for f in (lambda t: t, torch.abs))
    got = ops.indexed_inner_product(idx.cuda(), g.cuda(), src.cuda()).cpu().double()
    assert ((got - want).abs() <= (Dv + 8) * 2.0 ** -24 * scale).all()


# Rows' gradient where rows have few pairs: groups of 32 rows and what is left of one, empty rows, rows of 1, 32, 33 and hundreds of pairs,
# column passes, the average at and past the limit of 8 pairs a row
@pytest.mark.parametrize("B,I,rows,Dv", [(700, 32, 4007, 320), (512, 32, 2048, 192), (600, 32, 2048, 192), (96, 40, 3000, 1088)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rows_gradient_of_few_pairs(B, I, rows, Dv, dtype):
    gen = torch.Generator().manual_seed(B + I)
    idx = torch.randint(40, rows, (B, I), generator=gen, dtype=torch.int32)
    flat = idx.view(-1)
    flat[:600], flat[600:632], flat[632:665], flat[665] = 1, 2, 3, rows - 1
    g, w = torch.randn(B, Dv, generator=gen).to(dtype), torch.randn(B, I, generator=gen).to(dtype)
    want, scale = torch.zeros(rows, Dv, dtype=torch.double), torch.zeros(rows, Dv, dtype=torch.double)
    for i in range(I):
        products = w[:, i].double()[:, None] * g.double()
        want.index_add_(0, idx[:, i].long(), products)
        scale.index_add_(0, idx[:, i].long(), products.abs())
    got = ops.scatter_add(idx.cuda(), g.cuda(), w.float().cuda(), rows).cpu().double()
    n = torch.bincount(flat.long(), minlength=rows).double()[:, None]
    assert ((got - want).abs() <= (n + 4) * 2.0 ** -24 * scale).all()                # n additions in fp32


def _assert_same_infinities(got, want):
    got = torch.as_tensor(got).double()
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[got.isinf()], want[want.isinf()])


# Lists are padded to multiples of eight pairs: the padding adds nothing, not 0 * infinity.  By slices and by wavefronts, tokens that
# fill the copy of the gradient's last workgroup and a whole chunk of them
@pytest.mark.parametrize("B,I,rows,Dv", [(513, 62, 300, 320), (1024, 64, 300, 64), (16384, 8, 300, 64), (512, 32, 2048, 192)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rows_gradient_of_an_infinite_gradient(B, I, rows, Dv, dtype):
    gen = torch.Generator().manual_seed(B)
    idx = torch.randint(0, rows, (B, I), generator=gen, dtype=torch.int32)
    g, w = torch.randn(B, Dv, generator=gen).to(dtype), (0.1 + torch.rand(B, I, generator=gen)).to(dtype)
    g[0, 3], g[7, 5], g[B - 1, 0] = float("inf"), float("inf"), -float("inf")
    want = torch.zeros(rows, Dv, dtype=torch.double)
    for i in range(I):
        want.index_add_(0, idx[:, i].long(), w[:, i].double()[:, None] * g.double())
    src = torch.zeros(rows, Dv, dtype=dtype, device=DEV).requires_grad_()
    lookupffn_amd.weighted_gather_add(idx.to(DEV), src, w.to(DEV)).backward(g.to(DEV))
    _assert_same_infinities(src.grad.cpu(), want)


@pytest.mark.parametrize("B", [2500, 2560, 16384, 16385])
@pytest.mark.parametrize("S", [256, 512])
def test_tables_gradient_of_an_infinite_gradient(B, S):
    T, Do = 3, 64
    gen = torch.Generator().manual_seed(B)
    code = torch.randint(0, S, (B, T), generator=gen, dtype=torch.int32)
    score, g = 0.1 + torch.rand(B, T, generator=gen), torch.randn(B, Do, generator=gen)
    g[0, 3], g[64, 5], g[B - 1, 0] = float("inf"), float("inf"), -float("inf")
    want = torch.zeros(T, S, Do, dtype=torch.double)
    for t in range(T):
        want[t].index_add_(0, code[:, t].long(), score[:, t].double()[:, None] * g.double())
    _assert_same_infinities(cabi.lookup_scatter_sorted(code.numpy(), score.numpy(), g.numpy(), S), want)


# Rows of few tokens' gradients at and past the length from which a table's workgroups share a row out by columns: one slice of
# columns, uneven ones, several passes of one, tables of one and of several workgroups
@pytest.mark.parametrize("T,S,Do", [(3, 256, 64), (2, 256, 320), (1, 64, 832), (2, 256, 4672), (2, 16, 256)])
def test_gather_gradients_of_long_rows(T, S, Do):
    rng = np.random.RandomState(T + Do)
    lengths = [64, 65, 66, 200, 1]                                    # of rows 0, 1, 2, 9 and S - 1
    filled = np.repeat(np.array([0, 1, 2, 9, S - 1], np.int32), lengths)
    code = np.stack([rng.permutation(np.concatenate([filled, rng.randint(10, S, 700)])) for _ in range(T)], 1).astype(np.int32)
    B = len(code)
    score, g = rng.randn(B, T).astype(np.float32), rng.randn(B, Do).astype(np.float32)
    init = rng.randn(T, S, Do).astype(np.float32)
    want, scale = np.zeros((T, S, Do)), np.zeros((T, S, Do))
    for t in range(T):
        products = score[:, t, None].astype(np.float64) * g
        np.add.at(want[t], code[:, t], products)
        np.add.at(scale[t], code[:, t], np.abs(products))
    # products rounded to fp32, summed in fp64, the sum (and the one onto `init`) rounded to fp32
    assert (np.abs(cabi.lookup_scatter(code, score, g, S) - want) <= 2 * 2.0 ** -24 * scale).all()
    got = cabi.lookup_scatter(code, score, g, S, accumulate=True, init=init)
    assert (np.abs(got - want - init) <= 3 * 2.0 ** -24 * (scale + np.abs(init))).all()
