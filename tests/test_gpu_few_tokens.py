"""A token's columns shared out over several workgroups (csrc/token_gather.h): as from one, bit for bit."""
import ctypes
import math
from argparse import Namespace

import pytest
import torch

import lookupffn_amd
from lookupffn_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV, S = "cuda:0", 256


def _layer(H, D, R, T, Do, dtype, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(H + T + Do + seed)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    t = dict(ln_weight=1 + 0.1 * rand(H), ln_bias=0.1 * rand(H), diag=rand(R, 4, D) / math.sqrt(D), proj_bias=0.1 * rand(T * 8),
             tables=(0.02 * rand(T, S, Do)).to(dtype), out_bias=rand(Do))
    layer = _lib.FusedLayer(*(t[k].data_ptr() for k in ("ln_weight", "ln_bias", "diag", "proj_bias", "tables", "out_bias")),
                            H, D, R, 4, T, S, Do, 1e-5, 0.7, 0.3)
    return t, layer, rand


def _run(layer, fmt, x, residual, out):
    _lib.check(_lib.load().lffn_lookup_ffn_fused_layer_rows(ctypes.byref(layer), fmt, x.data_ptr(), _lib.ptr(residual), out.data_ptr(),
                                                            x.shape[0], _lib.stream_of(x)), "fused layer")
    return out


# 256 tokens have one workgroup each; fewer share out 2 to 10 passes of 256 columns, the last of them short, one and two passes to a workgroup
@pytest.mark.parametrize("H,D,R,T,Do,fmt", [(768, 1024, 1, 128, 768, 0), (500, 512, 2, 100, 260, 0), (256, 256, 1, 32, 516, 1),
                                            (1024, 1024, 2, 200, 1284, 2), (768, 1024, 1, 65, 2560, 0), (512, 512, 1, 64, 512, 2)])
def test_layer(H, D, R, T, Do, fmt):
    _, layer, rand = _layer(H, D, R, T, Do, [torch.float32, torch.bfloat16, torch.float16][fmt])
    x, residual = rand(256, H), rand(256, Do)
    want = _run(layer, fmt, x, residual, torch.full((256, Do), float("nan"), device=DEV))
    assert torch.isfinite(want).all()
    for B in (1, 17, 51, 64, 85, 86, 127, 128, 129):
        assert torch.equal(_run(layer, fmt, x[:B].clone(), residual[:B].clone(), torch.full((B, Do), float("nan"), device=DEV)), want[:B])
        again = residual[:B].clone()                      # the result in the residual's place
        assert torch.equal(_run(layer, fmt, x[:B].clone(), again, again), want[:B])


def test_result_in_the_input():
    """In the input's place a token's workgroup reads all it needs before it writes: one to a token then."""
    _, layer, rand = _layer(1024, 1024, 1, 128, 1024, torch.float32)
    x = rand(40, 1024)
    want = _run(layer, 0, x, x, torch.empty_like(x))
    assert torch.equal(_run(layer, 0, x, x, x), want)


@pytest.mark.parametrize("T,Do,fmt", [(128, 768, 0), (30, 1024, 1), (300, 576, 2)])
def test_gather_operators(T, Do, fmt):
    t, _, _ = _layer(64, 64, 1, T, Do, [torch.float32, torch.bfloat16, torch.float16][fmt])
    gen = torch.Generator(device=DEV).manual_seed(T)
    code = torch.randint(0, S, (256, T), generator=gen, device=DEV, dtype=torch.int32)
    score, tables = torch.rand(256, T, generator=gen, device=DEV), t["tables"]
    rows = (code + torch.arange(T, device=DEV, dtype=torch.int32) * S)[:, torch.randperm(T, generator=gen, device=DEV)].contiguous()
    want = ops.lookup_gather(code, score, tables, t["out_bias"]), ops.gather_add(rows, tables.view(T * S, Do), score)
    for B in (1, 63, 85, 128):
        assert torch.equal(ops.lookup_gather(code[:B], score[:B], tables, t["out_bias"]), want[0][:B])
        assert torch.equal(ops.gather_add(rows[:B], tables.view(T * S, Do), score[:B]), want[1][:B])


# either side of the line up to which the score gradient takes a token per workgroup
@pytest.mark.parametrize("T,Do,half", [(128, 1024, False), (30, 512, False), (64, 256, False), (60, 768, True), (33, 512, True)])
def test_inner_product_by_token_and_not(T, Do, half):
    """Sums of Do products, in any order: off by (Do + 1) 2^-24 of the magnitudes at most."""
    gen = torch.Generator(device=DEV).manual_seed(T + Do)
    last = min(1536, (768 if half else 384) * 1024 // Do)
    tables, g = 0.02 * torch.randn(T * S, Do, generator=gen, device=DEV), torch.randn(last + 1, Do, generator=gen, device=DEV)
    if half:
        tables, g = tables.half(), g.half()
    rows = torch.randint(0, S, (last + 1, T), generator=gen, device=DEV, dtype=torch.int32) + torch.arange(T, device=DEV, dtype=torch.int32) * S
    for B in (last, last + 1):
        got = ops.indexed_inner_product(rows[:B].contiguous(), g[:B].contiguous(), tables)
        for t in range(0, T, 7):
            term = tables[rows[:B, t].long()].double() * g[:B].double()
            assert ((got[:, t].double() - term.sum(-1)).abs() <= (Do + 1) * 2.0 ** -24 * term.abs().sum(-1)).all()


# either side of the line up to which a layer is one launch: tokens, tables times columns, rows of 16 bits
@pytest.mark.parametrize("T,Do,dtype,most", [(128, 896, torch.float32, 768), (128, 960, torch.float32, 512), (64, 128, torch.float32, 768),
                                             (128, 896, torch.bfloat16, 1152), (120, 1024, torch.float16, 768)])
def test_layer_in_one_launch_and_not(T, Do, dtype, most):
    cfg = Namespace(hidden_size=300, ffn_num_table=T, ffn_table_size=S, layer_norm_eps=1e-5, projection_type="bh4", block_size=1)
    torch.manual_seed(Do)
    layer = lookupffn_amd.LookupFFN(cfg, Do).to(DEV).eval()
    layer.tables.data = layer.tables.data.to(dtype)
    x, residual = torch.randn(most + 1, 300, device=DEV), torch.randn(most + 1, Do, device=DEV)
    with torch.no_grad():
        want = layer._forward_operators(x, residual)
        for B in (most, most + 1):
            assert layer.can_fuse_layer(x[:B]) == (B == most)
            # the same products summed over the tables in another order: T 2^-24 of their magnitudes (some 0.02 T^0.5 and the residual)
            assert (layer(x[:B], residual=residual[:B]) - want[:B]).abs().max() <= 1e-5
