"""A module computes the same whether gradients are recorded or not."""
import math
from argparse import Namespace

import pytest
import torch
from torch.utils.checkpoint import checkpoint

import lookupffn_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(hidden, tables, block, out, training=True):
    torch.manual_seed(hidden + tables)
    cfg = Namespace(hidden_size=hidden, ffn_num_table=tables, ffn_table_size=256, layer_norm_eps=1e-5, projection_type="bh4", block_size=block)
    layer = lookupffn_amd.LookupFFN(cfg, out).to(DEV).train(training)
    with torch.no_grad():
        layer.hash.projection.bias.normal_(std=0.05)
        if block == 1:
            layer.hash.projection.weight.copy_(layer.hash.projection.weight.sign() / math.sqrt(layer.hash.projection.padded_in_dim))
    return layer


def _same_rows(a, b):
    # sums over the tables in another order, either sign: 1e-6 of the results' size; another table row moves one by some 0.1
    return (a - b).abs().max().item() <= 1e-5 * b.pow(2).mean().sqrt().item()


# every form of the fp32 block kernel and of the diagonal one: few and many workgroups, one and several repeats, short rows.  The last
# size has 17 million projected values, a few of them within rounding of zero.
@pytest.mark.parametrize("tokens,hidden,tables,block", [(17, 256, 128, 64), (300, 512, 64, 64), (2103, 500, 128, 64), (3000, 1024, 32, 64),
                                                        (65, 64, 32, 64), (40, 256, 32, 1), (1500, 768, 128, 1), (16384, 512, 128, 64)])
@pytest.mark.parametrize("training", [True, False])
def test_a_layer_with_and_without_gradients(tokens, hidden, tables, block, training):
    layer = _layer(hidden, tables, block, 64, training)
    x = torch.randn(tokens, hidden, device=DEV)
    code, score = layer.hash(x)
    out = layer(x)
    assert score.requires_grad and out.requires_grad
    with torch.no_grad():
        plain = layer.hash(x)
        assert torch.equal(code, plain[0]) and torch.equal(score, plain[1])
        assert _same_rows(layer(x), out)
        assert _same_rows(layer._forward_operators(x, None), out)
    again = checkpoint(layer, x.clone().requires_grad_(), use_reentrant=True)
    assert again.requires_grad and _same_rows(again, out)


@pytest.mark.parametrize("training", [True, False])
def test_the_folded_blocks_follow_the_weights(training):
    layer = _layer(256, 32, 64, 64, training)
    x = torch.randn(50, 256, device=DEV)
    with torch.no_grad():
        for change in (lambda: None, lambda: layer.hash.projection.weight.mul_(1.5), lambda: layer.train(not training).train(training)):
            change()
            assert _same_rows(layer(x), layer._forward_operators(x, None))
            kept = layer.hash.__dict__.get("_folded")
            assert kept is not None and kept[1] is layer.hash.split_weight()


def test_only_the_copy_asked_for_is_folded(monkeypatch):
    """One launch after a change of the weights, whoever asks; another caller's copy beside it, and both follow the weights."""
    layer, made = _layer(256, 32, 64, 64, False), []
    for name in ("bh4_fold", "bh4_fold_split"):
        monkeypatch.setattr(lookupffn_amd.ops, name, lambda *a, name=name, fold=getattr(lookupffn_amd.ops, name): made.append(name) or fold(*a))
    x = torch.randn(50, 256, device=DEV)
    with torch.no_grad():
        for _ in range(2):
            layer(x), layer(x), layer._forward_operators(x, None)
            assert made == ["bh4_fold_split"]
            w = layer.hash.folded_weight()
            assert layer.hash.folded_weight() is w and made == ["bh4_fold_split", "bh4_fold"]
            assert torch.equal(w, lookupffn_amd.ops.bh4_fold_mode(layer.hash.projection.weight, 0).view_as(w))
            assert layer.hash.split_weight().numel() == lookupffn_amd.ops.split_words(layer.hash.projection.weight.shape)
            layer(x)
            assert len(made) == 2
            layer.hash.projection.weight.mul_(1.5)
            del made[:]
        state = layer.hash.__getstate__()
        assert not any(name.startswith("_folded") for name in state)
        layer.hash.invalidate_folded_weight()
        layer(x), layer.hash.folded_weight()
        assert made == ["bh4_fold_split", "bh4_fold"]


def test_an_encoder_layer_in_train_with_and_without_gradients():
    torch.manual_seed(1)
    cfg = Namespace(hidden_size=256, num_attention_heads=4, attention_head_size=64, attention_probs_dropout_prob=0.0, hidden_dropout_prob=0.0,
                    layer_norm_eps=1e-5, ffn_num_table=64, ffn_table_size=256, projection_type="bh4", block_size=1)
    layer = lookupffn_amd.EncoderLayer(cfg).to(DEV).train()
    x, mask = torch.randn(8, 300, 256, device=DEV), torch.ones(8, 300, device=DEV)
    mask[3, 200:] = 0
    half, out = layer.attention(x, mask), layer(x, mask)
    with torch.no_grad():
        assert torch.equal(layer.attention(x, mask), half)
        assert _same_rows(layer(x, mask), out)
    again = checkpoint(layer, x.clone().requires_grad_(), mask, use_reentrant=True)
    assert again.requires_grad and _same_rows(again, out)
