"""The sorted accumulation on top of what the rows hold: the sums are those of the plain call, added once, and rows that no token
points at are not touched."""
import ctypes

import numpy as np
import pytest
import torch

from lookupffn_amd import _lib
from tests import _cabi as cabi

pytestmark = pytest.mark.gpu
LIST_TOKENS = 2048                                      # LFFN_SCATTER_LIST_TOKENS


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


# 128 MiB of rows and more are stored past the caches, by each of the kernels that sum them: lists, the sorted accumulation in one chunk and
# in two, the sums of few and of many pairs
@pytest.mark.parametrize("B,T,Do", [(9, 256, 512), (2100, 256, 512), (16390, 256, 512), (9, 250, 512)])
def test_rows_written_past_the_caches(B, T, Do):
    gen = torch.Generator(device="cuda").manual_seed(B + T)
    code = torch.randint(0, 256, (B, T), generator=gen, device="cuda", dtype=torch.int32)
    code[:, 5] = 7                                      # a row of many pairs
    g, score = torch.randn(B, Do, generator=gen, device="cuda"), torch.rand(B, T, generator=gen, device="cuda")
    flat = code + 256 * torch.arange(T, device="cuda", dtype=torch.int32)
    layer = torch.full((T, 256, Do), float("nan"), device="cuda")
    cabi._call("lffn_lookup_scatter_f32", code.data_ptr(), score.data_ptr(), g.data_ptr(), layer.data_ptr(), B, T, 256, Do, 0)
    outs = [layer]
    size = ctypes.c_int64()
    if B > LIST_TOKENS:
        _lib.load().lffn_lookup_scatter_workspace_bytes(B, T, 256, Do, ctypes.byref(size))
        ws, out = torch.empty(size.value, dtype=torch.uint8, device="cuda"), torch.full_like(layer, float("nan"))
        cabi._call("lffn_lookup_scatter_sorted_f32", code.data_ptr(), score.data_ptr(), g.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, T,
                   256, Do, 0)
        outs.append(out)
    assert _lib.load().lffn_scatter_rows_workspace_bytes(B, T, T * 256, Do, ctypes.byref(size)) == 0
    if size.value > 0:
        ws, out = torch.empty(size.value, dtype=torch.uint8, device="cuda"), torch.full_like(layer, float("nan"))
        cabi._call("lffn_scatter_rows", flat.data_ptr(), g.data_ptr(), score.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel(), B, T, T * 256, Do,
                   0, 0)
        outs.append(out)
    for t in range(T):
        want, scale = (torch.zeros(256, Do, device="cuda", dtype=torch.float64) for _ in range(2))
        part = score[:, t:t + 1].double() * g.double()
        want.index_add_(0, code[:, t].long(), part)
        scale.index_add_(0, code[:, t].long(), part.abs())
        for out in outs:                                # fp32 sums of at most B products
            assert ((out[t] - want).abs() <= (B + 4) * 2.0 ** -24 * scale).all(), t

