"""The layer's host path (csrc/host.cpp) takes what it computes with from the layer on every call: a layer that was called before
and then changed is compared with one that was changed before its first call."""
import copy
import sys
import threading
import time
from argparse import Namespace

import pytest
import torch
import torch.autograd.forward_ad as fwAD

import lookupffn_amd
from lookupffn_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(block=1, seed=0, hidden=256, tables=32, out=256):
    torch.manual_seed(seed)
    cfg = Namespace(hidden_size=hidden, ffn_num_table=tables, ffn_table_size=256, layer_norm_eps=1e-5, projection_type="bh4",
                    block_size=block)
    layer = lookupffn_amd.LookupFFN(cfg, out).to(DEV)
    with torch.no_grad():
        for q in (layer.LayerNorm.weight, layer.LayerNorm.bias, layer.hash.projection.bias):
            q.add_(0.1 * torch.randn_like(q))
    return layer


def _pass(layer, x, train):
    """The result and, in training, the gradient of every parameter."""
    if not train:
        with torch.no_grad():
            return [layer.eval()(x)]
    layer.train().zero_grad(set_to_none=True)
    out = layer(x)
    out.sum().backward()
    return [out.detach()] + [q.grad for q in layer.parameters()]


def _assert_same(got, want):
    # (the two may take different kernels, whose fp32 sums of up to a few hundred terms are in another order)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5 * b.abs().max().item())


class Shifted(torch.nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner
        self.shift = torch.nn.Parameter(torch.full((inner.out_dim,), 0.3, device=DEV))

    def forward(self, x):
        return self.inner(x) + self.shift


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("block", [1, 64])
@pytest.mark.parametrize("which", ["LayerNorm", "hash", "projection", "wrapped projection"])
def test_replaced_modules_are_seen(block, train, which):
    layer, fresh, other = _layer(block), _layer(block), _layer(block, seed=1)
    x = torch.randn(40, 256, device=DEV)
    before = [_pass(layer, x, train) for _ in range(2)][0]
    for m in (layer, fresh):
        donor = copy.deepcopy(other)
        if which == "LayerNorm":
            m.LayerNorm = donor.LayerNorm
        elif which == "hash":
            m.hash = donor.hash
        elif which == "projection":
            m.hash.projection = donor.hash.projection
        else:
            m.hash.projection = Shifted(m.hash.projection)
    got = _pass(layer, x, train)
    assert not torch.allclose(got[0], before[0], rtol=1e-2)
    _assert_same(got, _pass(fresh, x, train))


@pytest.mark.parametrize("block", [1, 64])
def test_a_copy_with_parameters_of_its_own_uses_them(block):
    """A replica as DataParallel makes one shares the instance dictionary's entries but has other tensors as its parameters."""
    layer, other = _layer(block).eval(), _layer(block, seed=1).eval()
    x = torch.randn(40, 256, device=DEV)
    with torch.no_grad():
        layer(x), layer(x)
        replica = layer._replicate_for_data_parallel()
        replica._parameters = dict(other._parameters)
        replica._modules["LayerNorm"], replica._modules["hash"] = other.LayerNorm, other.hash
        _assert_same([replica(x)], [other(x)])
        assert torch.equal(layer(x), copy.deepcopy(layer)(x))


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("block", [1, 64])
@pytest.mark.parametrize("which", ["LayerNorm", "tables", "rows", "bias", "projection.bias", "projection"])
def test_parameters_that_do_not_fit_together_are_refused(block, train, which):
    """Each is one that the kernels, which take their sizes from the layer, would read beyond the end of."""
    layer = _layer(block)
    x = torch.randn(40, 256, device=DEV)
    _pass(layer, x, train), _pass(layer, x, train)
    zeros = lambda *shape: torch.nn.Parameter(torch.zeros(*shape, device=DEV))
    if which == "LayerNorm":
        layer.LayerNorm = torch.nn.LayerNorm(128).to(DEV)
    elif which == "tables":
        layer.tables = zeros(16, 256, 256)
    elif which == "rows":
        layer.tables = zeros(32, 128, 256)
    elif which == "bias":
        layer.bias = zeros(64)
    elif which == "projection.bias":
        layer.hash.projection.bias = zeros(128)
    else:
        layer.hash.projection = lookupffn_amd.BH4(128, 128, block).to(DEV)
    if which == "rows":          # a table of half as many rows is in order, and its rows are taken by the code's low bits
        assert torch.equal(_pass(layer, x, train)[0], layer.bias.detach().expand(40, 256))
        return
    with pytest.raises((AssertionError, RuntimeError)):
        _pass(layer, x, train)
        torch.cuda.synchronize()


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("block", [1, 64])
def test_changed_constants_are_seen(block, train):
    """A schedule on decay_coeff, another eps: the values the modules hold at the call."""
    layer, fresh = _layer(block), _layer(block)
    x = 0.01 * torch.randn(40, 256, device=DEV)                   # (small enough for eps to show)
    last = _pass(layer, x, train)
    for eps, decay in ((1e-3, 0.7), (1e-3, 0.4), (1, 1)):
        for m in (layer, fresh):
            m.LayerNorm.eps, m.hash.projection.decay_coeff = eps, decay
        got = _pass(layer, x, train)
        assert not torch.allclose(got[0], last[0], rtol=1e-2)
        _assert_same(got, _pass(copy.deepcopy(fresh), x, train))
        last = got


@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("block", [1, 64])
@pytest.mark.parametrize("name", ["tables", "bias", "LayerNorm.weight", "LayerNorm.bias", "hash.projection.weight",
                                  "hash.projection.bias"])
def test_a_tangent_on_a_parameter_is_refused(block, name, first):
    """As one on the input is, rather than dropped: the layer's autograd functions have no forward mode."""
    layer = _layer(block)
    x = torch.randn(20, 256, device=DEV)
    if not first:
        want = layer(x).detach()
        assert torch.equal(layer(x), want)
    params = dict(layer.named_parameters())
    with fwAD.dual_level():
        params[name] = fwAD.make_dual(params[name].detach(), torch.ones_like(params[name]))
        with pytest.raises((NotImplementedError, RuntimeError)):
            torch.func.functional_call(layer, params, (x,))
    if not first:
        assert torch.equal(layer(x), want)


@pytest.mark.parametrize("block", [1, 64])
def test_a_graph_through_the_gradients_ends_in_an_error(block):
    """create_graph: the gradients are the ones of an ordinary backward; a penalty on one of them raises, where it would
    have added nothing.  The residual's gradient is the result's and can be differentiated."""
    layer = _layer(block)
    x, res = torch.randn(20, 256, device=DEV, requires_grad=True), torch.randn(20, 256, device=DEV, requires_grad=True)
    inputs = [x, *layer.parameters()]
    want = torch.autograd.grad(layer(x).square().sum(), inputs)
    out = layer(x)
    got = torch.autograd.grad(out.square().sum(), inputs, create_graph=True)
    for a, b in zip(got, want):
        assert a.requires_grad and torch.equal(a.detach(), b)
        with pytest.raises(RuntimeError, match="differentiated"):
            (out.sum() + a.square().sum()).backward(retain_graph=True)
        with pytest.raises(RuntimeError, match="differentiated"):
            torch.autograd.grad(a.sum(), inputs, allow_unused=True, retain_graph=True)
    g, = torch.autograd.grad(layer(x, res).square().sum(), res, create_graph=True)
    g.sum().backward()
    assert torch.allclose(res.grad, torch.full_like(res, 2.0))


@pytest.mark.parametrize("how", ["class", "layer", "patched"])
def test_an_overridden_forward_is_called_every_time(how, monkeypatch):
    calls, base = [], lookupffn_amd.LookupFFN._forward

    def override(self, x, residual=None):
        calls.append((tuple(x.shape), residual is not None))
        return base(self, x, residual)

    layer = _layer().eval()
    x = torch.randn(2, 20, 256, device=DEV)
    with torch.no_grad():
        want = layer(x)
        if how == "class":
            layer.__class__ = type("Sub", (lookupffn_amd.LookupFFN,), {"_forward": override})
        elif how == "layer":
            layer._forward = lambda x, residual=None: override(layer, x, residual)
        else:
            monkeypatch.setattr(lookupffn_amd.LookupFFN, "_forward", override)
        for _ in range(3):
            assert torch.equal(layer(x), want)
        layer(x, x)
    assert calls == 3 * [((40, 256), False)] + [((40, 256), True)]


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("block", [1, 64])
def test_nothing_of_a_layer_is_held_between_calls(block, train):
    """Replaced parameters are freed at once, and torch.utils.swap_tensors, which wants no other reference, works."""
    layer = _layer(block)
    x = torch.randn(40, 256, device=DEV)
    _pass(layer, x, train), _pass(layer, x, train)
    layer.zero_grad(set_to_none=True)
    for name in ("tables", "bias"):
        torch.utils.swap_tensors(getattr(layer, name), torch.nn.Parameter(torch.ones_like(getattr(layer, name))))
    for m in (layer.LayerNorm, layer.hash.projection):
        torch.utils.swap_tensors(m.weight, torch.nn.Parameter(m.weight.detach().clone()))
    with torch.no_grad():
        code, score = layer.hash(layer.LayerNorm(x))
    _assert_same([_pass(layer, x, train)[0]], [(score.sum(1) + 1)[:, None].expand(40, 256)])
    layer.zero_grad(set_to_none=True)
    before, size = torch.cuda.memory_allocated(), layer.tables.numel() * 4
    layer.tables = None
    assert torch.cuda.memory_allocated() <= before - size


def test_inputs_as_a_caller_has_them():
    """Layouts of the input, shapes and types of the residual: the gradients and results of contiguous fp32 ones."""
    layer = _layer(out=128)
    x, res = torch.randn(6, 10, 256, device=DEV), torch.randn(6, 10, 128, device=DEV)
    g = torch.randn(6, 10, 128, device=DEV)

    def run(x, res):
        leaves = [t.detach().clone(memory_format=torch.preserve_format).requires_grad_() for t in (x, res)]
        out = layer(*leaves)
        assert out.shape == x.shape[:-1] + (128,) and out.is_contiguous()
        return [out.detach(), *torch.autograd.grad(out, [*leaves, layer.tables], g.reshape(out.shape))]

    want = run(x, res)
    strided = torch.empty(10, 6, 256, device=DEV).transpose(0, 1).copy_(x)
    for a, b in ((strided, res), (x, res.reshape(60, 128)), (x, res.double()), (strided, res.to(torch.float64).reshape(-1))):
        got = run(a, b)
        assert got[2].shape == b.shape and got[2].dtype == b.dtype
        for p, q in zip(got, want):
            assert torch.equal(p.reshape(q.shape).float(), q)
    half = run(x, res.to(torch.bfloat16))
    _assert_same(half[:1], run(x, res.to(torch.bfloat16).float())[:1])
    with torch.no_grad():
        assert torch.allclose(layer(strided, res), want[0], rtol=1e-4, atol=1e-5)
        with pytest.raises(RuntimeError):
            layer(x, res[:5])


@pytest.mark.parametrize("kind", ["taken", "dense projection", "fp64", "watched", "overridden"])
def test_the_host_path_is_tried_once_a_call(kind, monkeypatch):
    layer = _layer().eval()
    x = torch.randn(20, 256, device=DEV)
    if kind == "dense projection":
        layer.hash.projection = torch.nn.Linear(256, 256).to(DEV)
    elif kind == "fp64":
        layer, x = layer.double(), x.double()
    elif kind == "overridden":
        layer.__class__ = type("Sub", (lookupffn_amd.LookupFFN,), {"_forward": lambda self, *a: super(type(self), self)._forward(*a)})
    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    tries, real = [], _lib.host().forward

    class Counted:
        @staticmethod
        def forward(*args):
            out = real(*args)
            tries.append(out is not None)
            return out

    monkeypatch.setattr(_lib, "loaded_host", Counted)
    with torch.no_grad():
        for _ in range(2):
            if kind == "watched":
                with Watch():
                    layer(x)
            elif kind == "fp64":                       # (which the operators refuse)
                with pytest.raises((AssertionError, RuntimeError)):
                    layer(x)
            else:
                layer(x)
    assert tries == 2 * [kind in ("taken", "overridden")]


def test_other_threads_run_while_a_call_waits():
    """An allocation that has to go to the driver takes long enough for a thread that waits for the interpreter to get it."""
    layer = _layer(hidden=1024).eval()
    x = torch.randn(8192, 1024, device=DEV)
    count, stop, interval = [0], threading.Event(), sys.getswitchinterval()

    def spin():
        while not stop.is_set():
            count[0] += 1
            time.sleep(0)

    thread, moved = threading.Thread(target=spin), []
    with torch.no_grad():
        layer(x)
        try:
            sys.setswitchinterval(1.0)           # (nothing but a release gives the interpreter away)
            thread.start()
            for _ in range(20):
                torch.cuda.synchronize()
                torch.cuda.empty_cache()
                before = count[0]
                layer(x)
                moved.append(count[0] > before)
        finally:
            stop.set()
            sys.setswitchinterval(interval)
            thread.join()
    assert sum(moved) >= 10


def test_threads_and_streams_of_their_own():
    """Calls of several threads on one layer, each on a stream of its own, inference and training: every one's result."""
    layer = _layer()
    inputs = [torch.randn(40 * (i + 1), 256, device=DEV) for i in range(4)]
    with torch.no_grad():
        want = [layer(x) for x in inputs]
    torch.cuda.synchronize()
    failed = []

    def work(i):
        x = inputs[i].clone().requires_grad_()
        with torch.cuda.stream(torch.cuda.Stream()):
            torch.cuda.synchronize()
            for _ in range(30):
                with torch.no_grad():
                    out = layer(x)
                grad, = torch.autograd.grad(layer(x).sum(), x)
                torch.cuda.current_stream().synchronize()
                if not (torch.equal(out, want[i]) and torch.isfinite(grad).all()):
                    failed.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("block", [1, 64])
def test_a_layer_without_the_host_path_gives_the_same(block, train, monkeypatch):
    layer = _layer(block)
    x = torch.randn(40, 256, device=DEV)
    want = [t.clone() for t in _pass(layer, x, train)]
    monkeypatch.setattr(_lib, "loaded_host", False)
    _assert_same(_pass(layer, x, train), want)


def test_folded_blocks_are_those_of_the_weight_the_layer_has():
    """A weight that takes the address and the version number of one that was freed is another weight."""
    layer, fresh = _layer(64).eval(), _layer(64).eval()
    x = torch.randn(40, 256, device=DEV)
    p = layer.hash.projection
    new = torch.randn(p.weight.shape) / 128
    with torch.no_grad():
        layer(x)
        address, p.weight = p.weight.data_ptr(), None
        tries = [new.to(DEV)]
        while tries[-1].data_ptr() != address and len(tries) < 64:
            tries.append(new.to(DEV))
        p.weight = torch.nn.Parameter(tries[-1])
        fresh.hash.projection.weight = torch.nn.Parameter(new.to(DEV))
        assert torch.equal(layer(x), fresh(x))
        for a, b in zip(layer.hash(x), fresh.hash(x)):
            assert torch.equal(a, b)
        twin = copy.deepcopy(layer)
        assert "_folded" not in twin.hash.__dict__            # (it names an address of the other layer's)
        assert torch.equal(twin(x), layer(x))


@pytest.fixture(params=[True, False], ids=["host", "operators"])
def either_path(request, monkeypatch):
    if not request.param:
        monkeypatch.setattr(_lib, "loaded_host", False)


def test_folded_blocks_of_a_capture(either_path):
    """What a capture folds is not there before a replay, and its replays take the weights as they are then."""
    x = torch.randn(300, 256, device=DEV)
    with torch.no_grad():
        want = _layer(64).eval()(x)                           # (a layer of the same weights)
        layer = _layer(64).eval()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            static = layer(x)
        assert torch.equal(layer(x), want)
        for _ in range(4):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(static, layer(x))
            layer.hash.projection.weight.mul_(0.75)
            layer.hash.invalidate_folded_weight()
            junk = [torch.full_like(layer.hash.projection.weight, float("nan")) for _ in range(8)]
    assert len(junk) == 8


@pytest.mark.parametrize("block", [1, 64])
def test_a_compiled_layer(block):
    x = torch.randn(300, 256, device=DEV)
    layer = _layer(block).eval()
    compiled = torch.compile(layer, backend="eager")
    with torch.no_grad():
        for _ in range(2):                                    # (one launch and two may differ in the order of their sums)
            assert torch.allclose(compiled(x), layer(x), rtol=1e-5, atol=1e-6)
            layer.hash.projection.weight.mul_(0.75)


def test_folded_blocks_made_on_another_stream(either_path):
    """A call on another stream waits for them, and they stay until it has read them."""
    x = torch.randn(300, 256, device=DEV)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.no_grad():
        want = _layer(64).eval()(x)
        layer = _layer(64).eval()
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            torch.cuda._sleep(20_000_000)                     # some 10 to 200 ms
            layer(x)
        with torch.cuda.stream(second):
            got = layer(x)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        with torch.cuda.stream(second):
            torch.cuda._sleep(20_000_000)
            got = layer(x)
        with torch.cuda.stream(first):
            layer.hash.invalidate_folded_weight()
            junk = [torch.full_like(layer.hash.projection.weight, float("nan")) for _ in range(8)]
        torch.cuda.synchronize()
        assert torch.equal(got, want) and len(junk) == 8


# The backward exists twice, as one node in C++ and as the operators' autograd functions: at sizes where the forms of a kernel change
# (few tokens' gradients to 384, one-launch column sums to 1024 rows, lists to 2048, the sorted scatter and its chunks), for every
# gradient and for each one alone
@pytest.mark.parametrize("block,B,H,T,out", [(1, 1, 256, 32, 64), (64, 1, 256, 32, 64), (1, 384, 252, 34, 320), (64, 385, 512, 64, 512),
                                             (64, 1025, 700, 33, 192), (1, 2048, 1024, 128, 256), (1, 2049, 768, 128, 768),
                                             (64, 4097, 768, 128, 768), (1, 16385, 512, 32, 768)])
def test_both_backward_chains_agree(block, B, H, T, out, monkeypatch):
    layer = _layer(block, hidden=H, tables=T, out=out).train()
    gen = torch.Generator(device=DEV).manual_seed(B)
    x, res, g = (torch.randn(B, n, device=DEV, generator=gen) for n in (H, out, out))

    def run(wanted):
        leaves = dict(x=x.clone(), residual=res.clone(), **dict(layer.named_parameters()))
        for name, t in leaves.items():
            t.requires_grad_(wanted in (name, "all"))
        result = layer(leaves["x"], leaves["residual"])
        names = [name for name, t in leaves.items() if t.requires_grad]
        return dict(zip(["out", *names], [result.detach(), *torch.autograd.grad(result, [leaves[n] for n in names], g)]))

    wanted = ["all"] + (["x", "residual"] + [n for n, _ in layer.named_parameters()] if B < 5000 else [])
    host = [run(w) for w in wanted]
    monkeypatch.setattr(_lib, "loaded_host", False)
    for w, got in zip(wanted, host):
        want = run(w)
        assert got.keys() == want.keys()
        for name in want:
            # the same kernels; sums over the tokens that workgroups add up in the order they end differ in fp32's last bits
            assert (got[name] - want[name]).abs().max() <= 2e-6 * want[name].abs().max() + 1e-30, (w, name)
