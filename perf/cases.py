"""Performance cases: the work a program that uses this package has it do, through its public entry points.

Four kinds of pass:

  infer    LookupFFN.eval() without gradient on a batch of sequences (serving, evaluation), with or without the
           encoder's residual added inside, on fp32, bfloat16 or half tables, diagonal BH4 or 64 x 64 blocks
  train    LookupFFN.train(): forward, backward, the gradients of the input and of every parameter
  gather   weighted_gather_add, the operator, forward and backward, on flat row numbers: as LookupFFN.gather forms
           them (column i of the index array stays inside table i) or anywhere in the source; fp32 or all half
  encoder  EncoderLayer.eval(): attention and LookupFFN with their residuals, the layer a model is a stack of (one layer,
           since a second one turns rounding differences of the first into other table rows)

Ranges: 1 to 32768 tokens, hidden sizes from 256 to 1024 in steps of 64, 32 to 512 tables of 256 rows (the table size
of every configuration of this framework).
"""
import math
from argparse import Namespace

import torch

import lookupffn_amd

ROWS = 256                      # rows per table: 8-bit codes
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
INFER_MOST = 16384 * 512 * 1024          # (token, table, column) products of the largest case of a kind
TRAIN_MOST = 32768 * 128 * 512
GATHER_MOST = 4096 * 128 * 512
ENCODER_MOST = 16384 * 768


def listed():
    infer = dict(kind="infer", tables="f32", block=1, residual=False)
    train = dict(kind="train", block=1)
    return [
        # one short sentence through a RoBERTa-base layer: nothing but launch latency and a chain of memory round trips
        dict(infer, name="infer-17-base", batch=1, seq=17, hidden=768, num_table=128),
        # the smallest configuration of the benchmark: 2 x 128 tokens, 32 tables
        dict(infer, name="infer-256-small", batch=2, seq=128, hidden=256, num_table=32),
        # a batch of sentences cut to their longest, inside an encoder layer: ragged, too few tokens to fill the chip easily
        dict(infer, name="infer-2103-base-residual", batch=3, seq=701, hidden=768, num_table=128, residual=True),
        # the benchmark's default: 32 x 512 tokens at the RoBERTa-base layer
        dict(infer, name="infer-16384-base", batch=32, seq=512, hidden=768, num_table=128),
        # the layer of the reference's training configurations and timing script: hidden 512, 64 x 64 blocks, 64 x 512 tokens
        dict(infer, name="infer-32768-512-block64", batch=64, seq=512, hidden=512, num_table=128, block=64),
        # 512 tables of 1024 columns: fp32 tables beyond the memory-side cache, and the same in bfloat16
        dict(infer, name="infer-16384-large", batch=32, seq=512, hidden=1024, num_table=512),
        dict(infer, name="infer-16384-large-bf16", batch=32, seq=512, hidden=1024, num_table=512, tables="bf16"),
        # fine-tuning on a few sentences with the reference's second table count: a training step that is all latency
        dict(train, name="train-385-512-block64", batch=5, seq=77, hidden=512, num_table=64, block=64),
        # training steps at the RoBERTa-base layer and at the reference's own training configuration
        dict(train, name="train-16384-base", batch=32, seq=512, hidden=768, num_table=128),
        dict(train, name="train-32768-512-block64", batch=64, seq=512, hidden=512, num_table=128, block=64),
        # the operator the reference's module calls, used on its own in a training program
        dict(kind="gather", name="gather-4096-512", batch=4096, hidden=512, num_table=128, indexes="tables", dtype="f32"),
        # one of the twelve layers of the benchmark's RoBERTa-base encoder, 32 x 512 tokens
        dict(kind="encoder", name="encoder-16384-base", batch=32, seq=512, hidden=768, num_table=128, block=1),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _split(rng, tokens):
    """tokens as about that many in a batch of equal sequences of at most 512."""
    seq = min(tokens, _log_int(rng, 1, 512))
    return max(1, tokens // seq), seq


def draw(rng):
    kind = rng.choices(["infer", "train", "gather", "encoder"], [10, 6, 3, 1])[0]
    while True:
        hidden = rng.choice([256, 512, 768, 1024, 64 * rng.randint(4, 16)])
        num_table = rng.choice([32, 64, 128, 128, 256, 512])
        if kind == "infer":
            batch, seq = _split(rng, _log_int(rng, 1, 32768))
            case = dict(kind=kind, batch=batch, seq=seq, hidden=hidden, num_table=num_table, block=rng.choice([1, 1, 64]),
                        tables=rng.choice(["f32", "f32", "bf16", "f16"]), residual=rng.random() < 0.5)
            if batch * seq * num_table * hidden <= INFER_MOST:
                return case
        elif kind == "train":
            batch, seq = _split(rng, _log_int(rng, 64, 32768))
            case = dict(kind=kind, batch=batch, seq=seq, hidden=hidden, num_table=num_table, block=rng.choice([1, 64]))
            if batch * seq * num_table * hidden <= TRAIN_MOST:
                return case
        elif kind == "gather":
            batch = _log_int(rng, 64, 16384)
            case = dict(kind=kind, batch=batch, hidden=hidden, num_table=num_table, dtype=rng.choice(["f32", "f32", "f16"]),
                        indexes=rng.choice(["tables", "tables", "any"]))
            if batch * num_table * hidden <= GATHER_MOST:
                return case
        else:
            batch, seq = _log_int(rng, 1, 32), _log_int(rng, 16, 512)
            hidden, num_table = rng.choice([(512, 64), (512, 128), (768, 128)])
            case = dict(kind=kind, batch=batch, seq=seq, hidden=hidden, num_table=num_table, block=rng.choice([1, 64]))
            if batch * seq * hidden <= ENCODER_MOST:
                return case


def _config(case):
    return Namespace(hidden_size=case["hidden"], ffn_num_table=case["num_table"], ffn_table_size=ROWS, layer_norm_eps=1e-5,
                     projection_type="bh4", block_size=case["block"], num_attention_heads=case["hidden"] // 64,
                     attention_head_size=64, attention_probs_dropout_prob=0.1, hidden_dropout_prob=0.1)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


@torch.no_grad()
def _fill(layer, gen):
    """A layer's parameters, as initialised and moved a little by training; a diagonal projection starts from signs, so
    that its stages are orthonormal."""
    ln, p = layer.LayerNorm, layer.hash.projection
    ln.weight.copy_(1 + 0.1 * _randn(gen, *ln.weight.shape))
    ln.bias.copy_(0.1 * _randn(gen, *ln.bias.shape))
    w = _randn(gen, *p.weight.shape)
    if p.block_size == 1:
        w = torch.sign(w) + 0.05 * _randn(gen, *w.shape)
    p.weight.copy_(w / math.sqrt(p.block_size * p.padded_in_dim))
    p.bias.copy_(0.05 * _randn(gen, *p.bias.shape))
    layer.tables.copy_(0.02 * _randn(gen, *layer.tables.shape))
    layer.bias.copy_(0.001 * _randn(gen, *layer.bias.shape))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, hidden = case["kind"], case["hidden"]
    if kind == "gather":
        tokens, cols, dt = case["batch"], case["num_table"], DTYPES[case["dtype"]]
        rows = cols * ROWS
        if case["indexes"] == "tables":
            indexes = torch.randint(0, ROWS, (tokens, cols), generator=gen, device="cuda", dtype=torch.int32)
            indexes += torch.arange(cols, device="cuda", dtype=torch.int32)[None] * ROWS
        else:
            indexes = torch.randint(0, rows, (tokens, cols), generator=gen, device="cuda", dtype=torch.int32)
        source = (0.02 * _randn(gen, rows, hidden)).to(dt).requires_grad_()
        weights = (1 - torch.rand(tokens, cols, generator=gen, device="cuda")).to(dt).requires_grad_()
        return dict(kind=kind, indexes=indexes, source=source, weights=weights, grad=_randn(gen, tokens, hidden).to(dt))
    with torch.device("cuda"):
        model = (lookupffn_amd.EncoderLayer(_config(case)) if kind == "encoder" else
                 lookupffn_amd.LookupFFN(_config(case), hidden))
    batch, seq = case["batch"], case["seq"]
    x = _randn(gen, batch, seq, hidden)
    if kind == "encoder":
        with torch.no_grad():
            for linear in (model.attention.query, model.attention.key, model.attention.value, model.attention.dense):
                linear.weight.copy_(_randn(gen, hidden, hidden) / math.sqrt(hidden))
                linear.bias.copy_(0.05 * _randn(gen, hidden))
        _fill(model.FFN, gen)
        # a batch of sentences is padded to the longest: between none and a half of a sentence is padding
        length = torch.randint((seq + 1) // 2, seq + 1, (batch, 1), generator=gen, device="cuda")
        mask = (torch.arange(seq, device="cuda")[None] < length).float()
        return dict(kind=kind, model=model.eval(), x=x, mask=mask)
    _fill(model, gen)
    if kind == "train":
        return dict(kind=kind, layer=model.train(), x=x.requires_grad_(), grad=_randn(gen, batch, seq, hidden))
    if case["tables"] != "f32":
        model.tables.data = model.tables.data.to(DTYPES[case["tables"]])
    return dict(kind=kind, layer=model.eval(), x=x, residual=_randn(gen, batch, seq, hidden) if case["residual"] else None)


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            if state["residual"] is None:
                return state["layer"](state["x"])
            return state["layer"](state["x"], residual=state["residual"])
    if kind == "train":
        layer, x = state["layer"], state["x"]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        out = layer(x)
        out.backward(state["grad"])
        return dict(out=out.detach(), x=x.grad, **{name: p.grad for name, p in layer.named_parameters()})
    if kind == "gather":
        source, weights = state["source"], state["weights"]
        source.grad = weights.grad = None
        out = lookupffn_amd.weighted_gather_add(state["indexes"], source, weights)
        out.backward(state["grad"])
        return dict(out=out.detach(), source=source.grad, weights=weights.grad)
    with torch.no_grad():
        return state["model"](state["x"], state["mask"])


def _projection(case, tokens):
    """(weights, operations) of one forward projection of `tokens` rows."""
    dim = 2 ** math.ceil(math.log2(case["hidden"]))
    repeats = max(1, math.ceil(8 * case["num_table"] / dim))
    block = case["block"]
    per_stage = 2 * dim * block + dim * (math.log2(dim) if block == 1 else math.log2(dim / block))
    return 4 * repeats * dim * block, tokens * repeats * 4 * per_stage


def work(case):
    kind, hidden, tables = case["kind"], case["hidden"], case["num_table"]
    tokens = case["batch"] * case.get("seq", 1)
    products = 2 * tokens * tables * hidden
    touched = min(tables * ROWS, tokens * tables) * hidden        # elements of the rows that are read at all
    if kind == "gather":
        size = torch.finfo(DTYPES[case["dtype"]]).bits // 8
        # rows, indexes, weights and the gradient in; the result, the weights' gradient and the whole source gradient out
        moved = size * (touched + 2 * tokens * hidden + 2 * tokens * tables + tables * ROWS * hidden) + 4 * tokens * tables
        return {"bytes": moved, "flops": 3 * products}
    weights, operations = _projection(case, tokens)
    params = 4 * (weights + 3 * hidden + 8 * tables)
    if kind == "infer":
        size = torch.finfo(DTYPES[case["tables"]]).bits // 8
        moved = 4 * tokens * hidden * (3 if case["residual"] else 2) + params + size * touched
        return {"bytes": moved, "flops": products + operations}
    if kind == "train":
        # input, gradient of the output, rows read; output, gradients of the input and of every parameter written
        moved = 4 * tokens * hidden * 4 + 2 * params + 4 * touched + 4 * tables * ROWS * hidden
        return {"bytes": moved, "flops": 3 * (products + operations)}
    # the four matrices of the attention and its two products per head; hidden states in and out, the mask
    seq = case["seq"]
    attention = 8 * tokens * hidden * hidden + 4 * tokens * seq * hidden
    moved = params + 4 * touched + 16 * hidden * hidden + 4 * tokens * (2 * hidden + 1)
    return {"bytes": moved, "flops": products + operations + attention}


def tolerance(case):
    kind = case["kind"]
    if kind == "gather":
        # fp32 sums of products; an all-half call rounds its results to half
        return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 1e-3, "max": 1e-2}
    # A projected value within fp32 rounding (about 1e-6 of its spread) of zero takes either sign, and with the sign one of
    # the token's T rows is another one: sqrt(2 / T) of that token's result.  Per token 8 T values, so 8 T * 8e-7 rows
    # change and the whole result moves by sqrt(2 / T * 8 T * 8e-7) = 4e-3, whatever T; a small batch has to bear one
    # changed row in any case.
    tokens = case["batch"] * case["seq"]
    return {"rel": min(0.03, max(4e-3, math.sqrt(2 / (case["num_table"] * tokens)))), "max": 0.99}
