"""The gather whose table pairs are shared out over several workgroups (csrc/lookup_gather_quad.hip, lookup_gather.hip)."""
import ctypes
import sys

import pytest
import torch

from lookupffn_amd import _lib, ops

S = 256
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _plan(B, T, Do, fmt, packed):
    plan = _lib.GatherParts()
    assert _lib.load().lffn_lookup_gather_parts_plan(B, T, S, Do, fmt, packed, ctypes.byref(plan)) == 0
    return plan


def test_plans_fit_the_kernel():
    seen = 0
    for B in (1, 200, 1000, 2103, 4096, 5001, 8192, 12288, 16384, 100000):
        for T in (2, 7, 8, 64, 66, 128, 512):
            for Do in (64, 192, 512, 768, 1024, 4096):
                for fmt in (0, 1, 2):
                    for packed in (0, 1):
                        p = _plan(B, T, Do, fmt, packed)
                        if p.parts == 0:
                            assert p.bytes == 0 and p.tokens_per_workgroup == 0
                            continue
                        seen += 1
                        tile, pairs = p.tokens_per_workgroup, -(-T // 2 // p.parts)
                        assert T % 2 == 0 and tile % 16 == 0 and 768 < tile <= (1024 if fmt else 2048)
                        assert p.parts >= 2 and (p.parts - 1) * pairs < T // 2                      # no part is empty
                        tiles = -(-B // tile)
                        assert p.record_stride == tiles * tile and tiles * p.parts * Do * (2 if fmt else 4) // 128 <= 256
                        assert p.bytes == 6 * T * p.record_stride + 4 * p.parts * B * Do
    assert seen > 100


def test_refusals():
    lib, A, U, P = _lib.load(), _lib.LFFN_ERR_BAD_ARG, _lib.LFFN_ERR_UNSUPPORTED, 256
    call = lambda tile, parts, stride, code=P, score=P, out=P, ws=P, room=1 << 30, T=64, s=S: lib.lffn_lookup_gather_parts_rows(
        ctypes.byref(_lib.GatherParts(tile, parts, stride, 0)), code, score, P, None, None, out, ws, room, 1000, T, s, 512, 0, None)
    assert call(1000, 4, 1000) == A and call(1008, 0, 1008) == A and call(1008, 4, 1000) == A and call(1008, 4, 1010) == A
    assert call(512, 4, 1024) == U                       # two passes are not built
    assert call(1008, 4, 1008, T=63) == U and call(1008, 4, 1008, s=128) == U
    assert call(1008, 33, 1008) == U and call(1008, 31, 1008) == U             # 32 pairs: 33 parts, or 31 of two pairs
    assert call(1008, 4, 1008, code=None) == A and call(1008, 4, 1008, score=260) == A and call(1008, 4, 1008, code=260) == A
    assert call(1008, 4, 1008, out=264) == A and call(1008, 4, 1008, ws=264) == A and call(1008, 4, 1008, ws=None) == A
    assert call(1008, 4, 1008, room=6 * 64 * 1008 + 4 * 4 * 1000 * 512 - 1) == A
    assert lib.lffn_lookup_gather_parts_plan(1000, 64, S, 512, 3, 0, ctypes.byref(_lib.GatherParts())) == A


def _inputs(B, T, Do, fmt):
    gen = torch.Generator(device="cuda").manual_seed(B + T + Do)
    tables = (0.02 * torch.randn(T, S, Do, generator=gen, device="cuda")).to(DTYPES[fmt])
    code = torch.randint(0, S, (B, T), generator=gen, device="cuda", dtype=torch.int32)
    score, bias = torch.rand(B, T, generator=gen, device="cuda") - 0.3, torch.randn(Do, generator=gen, device="cuda")
    return tables, code, score, bias, torch.randn(B, Do, generator=gen, device="cuda")


def _check(out, tables, code, score, bias=None, residual=None):
    """Against 64 bits: T products and T + 2 additions, each off by 2^-24 of the sum of the magnitudes at most."""
    T = code.shape[1]
    want, size = (torch.zeros(out.shape, dtype=torch.float64, device="cuda") for _ in range(2))
    for t in range(T):
        term = tables[t].double()[code[:, t].long()] * score[:, t:t + 1].double()
        want += term
        size += term.abs()
    for extra in (bias, residual):
        if extra is not None:
            want += extra.double()
            size += extra.double().abs()
    assert ((out.double() - want).abs() <= (T + 3) * 2.0 ** -24 * size).all()


# tiles that end in a pass, in a wavefront's group and in a quad; parts of one pair, a short last part, two and many tiles
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,Do,fmt,tile,parts", [
    (1000, 8, 64, 0, 1008, 4), (1, 4, 64, 0, 784, 2), (2103, 26, 192, 0, 1056, 5), (777, 26, 32 * 6, 0, 1040, 3),
    (5000, 14, 128, 0, 1280, 3), (3001, 20, 128, 0, 1520, 4), (3001, 20, 128, 0, 1808, 10), (4099, 6, 64, 0, 2048, 2),
    (3200, 12, 64, 0, 800, 2), (1500, 10, 128, 1, 784, 5), (2050, 20, 192, 2, 1024, 4), (700, 12, 64, 1, 1024, 6),
    (900, 12, 64, 0, 912, 1)])
def test_parts_against_64_bits(B, T, Do, fmt, tile, parts):
    tables, code, score, bias, residual = _inputs(B, T, Do, fmt)
    stride = -(-B // tile) * tile
    room = 6 * T * stride + 4 * parts * B * Do
    plan = _lib.GatherParts(tile, parts, stride, room)

    def run(b, r, out, records=False):
        ws = torch.full((room // 4,), float("nan"), device="cuda") if not records else records[0]
        _lib.check(_lib.load().lffn_lookup_gather_parts_rows(
            ctypes.byref(plan), *(None, None) if records else (code.data_ptr(), score.data_ptr()), tables.data_ptr(), _lib.ptr(b),
            _lib.ptr(r), out.data_ptr(), ws.data_ptr(), room, B, T, S, Do, fmt, _lib.stream_of(out)), "parts")
        return ws

    out = torch.full((B, Do), float("nan"), device="cuda")
    ws = run(bias, residual, out)
    _check(out, tables, code, score, bias, residual)
    again = residual.clone()
    run(bias, again, again, records=(ws,))               # records that are there, the residual in the output's place
    assert torch.equal(out, again)
    run(None, None, out)
    _check(out, tables, code, score)


# by the callers' own choice: the layer's operator and the plain gather, whose row numbers are in table form or not
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,Do,fmt", [(3300, 128, 512, 0), (5000, 128, 768, 0), (6200, 128, 512, 1), (8000, 64, 1024, 2)])
def test_operators_take_it(B, T, Do, fmt):
    assert _plan(B, T, Do, fmt, 0).parts
    tables, code, score, bias, residual = _inputs(B, T, Do, fmt)
    _check(ops.lookup_gather(code, score, tables, bias, residual), tables, code, score, bias, residual)
    odd = torch.cat([code.new_zeros(1), code.flatten()])[1:].view(B, T)                             # 4 bytes off
    _check(ops.lookup_gather(odd, score, tables, bias), tables, code, score, bias)
    rows = code + torch.arange(T, device="cuda", dtype=torch.int32) * S
    flat = tables.view(T * S, Do)
    _check(ops.gather_add(rows, flat, score), tables, code, score)
    order = torch.randperm(T, device="cuda")
    rows[1], weights = rows[1, order], score.clone()                                                # one token out of table form
    weights[1] = score[1, order]
    _check(ops.gather_add(rows, flat, weights), tables, code, score)


# the benchmark times the layer's stages apart and asks for the layer's result bit for bit
@pytest.mark.gpu
@pytest.mark.parametrize("B,bs", [(6144, 1), (2103, 1), (4096, 64)])
def test_the_benchmarks_stages_are_the_layers(B, bs, monkeypatch, capsys):
    import bench
    assert _plan(B, 128, 768, 0, 1).parts
    monkeypatch.setitem(bench.WORKLOADS, "parts", dict(B=B, H=768, T=128, S=S, Do=768, bf16=False, bs=bs, desc=""))
    monkeypatch.setattr(sys, "argv", "bench.py --workload parts --steps 2 --warmup 1 --no-settle --no-cpu-baseline".split())
    bench.main()
    assert "of the tables per workgroup" in capsys.readouterr().out
