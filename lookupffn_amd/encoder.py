"""The caller of the hot path: the reference's pre-norm encoder with LookupFFN in
place of the feed-forward block (PL/layer.py, PL/encoder.py, and the embeddings
of src/roberta/models/postnorm.py:6-28), with the same module and parameter
names so that a reference state_dict loads unchanged.  ``LookupFFN`` and, without
gradients, the attention's products and softmax run on the gfx950 kernels of this
package; embeddings, LayerNorms and the attention in training are plain PyTorch-ROCm.

``config`` carries the attributes the reference reads: hidden_size,
num_attention_heads, attention_head_size, attention_probs_dropout_prob,
hidden_dropout_prob, layer_norm_eps, num_hidden_layers, vocab_size,
max_position_embeddings, type_vocab_size, pad_token_id, plus LookupFFN's
(ffn_num_table, ffn_table_size, projection_type, block_size) and optionally
checkpoint_attention.
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from . import ops
from .lookup import LookupFFN

_GLOBAL_HOOKS = torch.nn.modules.module
_FORWARDS = {kind: kind.forward for kind in (nn.Linear, nn.LayerNorm, nn.Dropout)}       # (and Attention, below)


def _plain(module, kind):
    """module is a `kind` itself, the class as it was written, and nothing watches its calls: what it computes may be computed
    without calling it."""
    return (type(module) is kind and "forward" not in module.__dict__ and kind.forward is _FORWARDS[kind]
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks))


def _nobody_watches():
    """No tracer, transform, mode or hook on every module has to see the operators one by one."""
    return not (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch.jit.is_scripting() or torch.is_autocast_enabled("cuda")
                or torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack() or torch.autograd.forward_ad._current_level >= 0
                or _GLOBAL_HOOKS._global_forward_hooks or _GLOBAL_HOOKS._global_forward_pre_hooks
                or _GLOBAL_HOOKS._global_backward_hooks or _GLOBAL_HOOKS._global_backward_pre_hooks)


def _kernel_operand(t, shape, device):
    return (type(t) in (torch.Tensor, nn.Parameter) and t.dtype == torch.float32 and t.device == device and t.shape == shape
            and t.is_contiguous() and t.data_ptr() % 16 == 0)


class RobertaEmbeddings(nn.Module):
    """word + token-type + position embeddings, LayerNorm, dropout
    (src/roberta/models/postnorm.py:6-28); positions are offset by pad_token_id + 1."""

    def __init__(self, config):
        super().__init__()
        self.pad_token_id = config.pad_token_id
        self.word_embeddings = nn.Embedding(config.vocab_size, config.hidden_size)
        self.position_embeddings = nn.Embedding(config.max_position_embeddings + 2, config.hidden_size)
        self.token_type_embeddings = nn.Embedding(config.type_vocab_size, config.hidden_size)
        self.LayerNorm = nn.LayerNorm(config.hidden_size, eps=config.layer_norm_eps)
        self.dropout = nn.Dropout(config.hidden_dropout_prob)

    def forward(self, input_ids, token_type_ids, position_ids):
        x = (self.word_embeddings(input_ids)
             + self.token_type_embeddings(token_type_ids)
             + self.position_embeddings(position_ids + (self.pad_token_id + 1)))
        return self.dropout(self.LayerNorm(x))


class Attention(nn.Module):
    """Pre-norm multi-head self-attention (PL/layer.py:11-64): LayerNorm, q/k/v
    projections, softmax(q k^T / sqrt(d) - 1000 * (1 - mask)) v in float32, output
    projection.  ``fused=True`` evaluates the same expression with
    scaled_dot_product_attention; ``fused=False`` is the reference's literal
    sequence of matmuls."""

    def __init__(self, config, fused=True):
        super().__init__()
        self.num_attention_heads = config.num_attention_heads
        self.attention_head_size = config.attention_head_size
        self.all_head_size = self.num_attention_heads * self.attention_head_size
        self.dropout = nn.Dropout(config.attention_probs_dropout_prob)
        self.checkpoint_attention = bool(getattr(config, "checkpoint_attention", False))
        self.fused = fused

        self.LayerNorm = nn.LayerNorm(config.hidden_size, eps=config.layer_norm_eps)
        self.query = nn.Linear(config.hidden_size, config.hidden_size)
        self.key = nn.Linear(config.hidden_size, config.hidden_size)
        self.value = nn.Linear(config.hidden_size, config.hidden_size)
        self.dense = nn.Linear(config.hidden_size, config.hidden_size)

    def transpose_for_scores(self, x):
        return x.view(*x.shape[:-1], self.num_attention_heads, self.attention_head_size).permute(0, 2, 1, 3)

    def attention(self, query_layer, key_layer, value_layer, attention_mask):
        bias = -1000.0 * (1.0 - attention_mask[:, None, None, :].float())
        q, k, v = query_layer.float(), key_layer.float(), value_layer.float()
        if self.fused:
            ctx = F.scaled_dot_product_attention(q, k, v, attn_mask=bias,
                                                 dropout_p=self.dropout.p if self.training else 0.0)
        else:
            scale = self.attention_head_size ** 0.25
            probs = torch.softmax(torch.matmul(q / scale, (k / scale).transpose(-1, -2)) + bias, dim=-1)
            ctx = torch.matmul(self.dropout(probs), v)
        return ctx.to(value_layer.dtype)

    def _kernels_apply(self, x, mask):
        """The products and the softmax go to this package's kernels (csrc/linear.hip, csrc/attention.hip): fp32 on the GPU in eval() without
        gradients, heads of 64 columns, and every part of the module the one it was built with.  A module in train() keeps the
        library's with and without gradients: a checkpointed pass runs both, and the LookupFFN behind turns a rounding into another
        table row.  Against the library's fp32
        products and attention the encoder layer takes, 32 x 512 tokens of 768, 624 us instead of 1279, 4 x 128 tokens 86 instead of
        164, 16 tokens 86 instead of 166, and its attention half is half as far from 64 bits (5e-7 against 9e-7)."""
        linears = (self.query, self.key, self.value, self.dense)
        if not (x.is_cuda and x.dim() == 3 and x.dtype == torch.float32 and x.numel() > 0 and type(x) in (torch.Tensor, nn.Parameter)
                and self.fused and not self.training and type(self) is Attention
                and not any(name in self.__dict__ or getattr(Attention, name) is not method for name, method in _OWN_METHODS)):
            return False
        hidden = x.shape[2]
        return (self.attention_head_size == 64 and self.all_head_size == hidden and x.shape[1] <= ops.ATTENTION_MAX_KEYS
                and type(mask) is torch.Tensor and mask.shape == x.shape[:2] and mask.device == x.device
                and all(_plain(m, nn.Linear) and _kernel_operand(m.weight, (hidden, hidden), x.device)
                        and (m.bias is None or _kernel_operand(m.bias, (hidden,), x.device)) for m in linears)
                and not (torch.is_grad_enabled()
                         and (x.requires_grad or mask.requires_grad or any(p.requires_grad for p in self.parameters())))
                and _nobody_watches())

    def _norm_applies(self, x):
        """The LayerNorm is the one the module was built with and there are rows enough that its kernel splits them, and the weights,
        once for all tiles."""
        norm, shape = self.LayerNorm, x.shape[2:]
        return (x.shape[0] * x.shape[1] >= ops.LINEAR_NORM_MIN_ROWS and shape[0] <= ops.LINEAR_NORM_MAX_COLUMNS
                and _plain(norm, nn.LayerNorm) and norm.normalized_shape == tuple(shape) and _kernel_operand(x, x.shape, x.device)
                and all(p is None or _kernel_operand(p, shape, x.device) for p in (norm.weight, norm.bias)))

    def _forward_kernels(self, hidden_states, attention_mask, residual=None):
        B, L, hidden = hidden_states.shape
        q, k, v, dense, norm = self.query, self.key, self.value, self.dense, self.LayerNorm
        weights, biases = (q.weight, k.weight, v.weight), (q.bias, k.bias, v.bias)
        if self._norm_applies(hidden_states):
            qkv = ops.linear_norm(hidden_states.view(B * L, hidden), norm.weight, norm.bias, float(norm.eps), weights, biases)
        else:
            h = norm(hidden_states)
            if not _kernel_operand(h, hidden_states.shape, hidden_states.device):        # another LayerNorm may return anything
                out = self._attend(h, attention_mask)
                return out if residual is None else out + residual
            qkv = ops.linear(h.view(B * L, hidden), weights, biases, None)
        qkv = qkv.view(3, B, L, self.num_attention_heads, 64)
        ctx = ops.attention(qkv[0], qkv[1], qkv[2], attention_mask.float().contiguous())
        if residual is not None:
            residual = residual.contiguous().view(B * L, hidden)
        return ops.linear(ctx.view(B * L, hidden), (dense.weight,), (dense.bias,), residual).view(B, L, hidden)

    def _attend(self, h, attention_mask):
        q = self.transpose_for_scores(self.query(h))
        k = self.transpose_for_scores(self.key(h))
        v = self.transpose_for_scores(self.value(h))
        if self.checkpoint_attention:
            ctx = checkpoint(self.attention, q, k, v, attention_mask, use_reentrant=False)
        else:
            ctx = self.attention(q, k, v, attention_mask)
        ctx = ctx.permute(0, 2, 1, 3).contiguous()
        return self.dense(ctx.view(*ctx.shape[:-2], self.all_head_size))

    def forward(self, hidden_states, attention_mask):
        if self._kernels_apply(hidden_states, attention_mask):
            return self._forward_kernels(hidden_states, attention_mask)
        return self._attend(self.LayerNorm(hidden_states), attention_mask)


# What the kernels stand in for: a class or a module with another one has it called.
_FORWARDS[Attention] = Attention.forward
_OWN_METHODS = tuple((name, getattr(Attention, name)) for name in ("attention", "transpose_for_scores", "_attend"))


class EncoderLayer(nn.Module):
    """attention + residual, LookupFFN + residual (PL/layer.py:66-78)."""

    def __init__(self, config):
        super().__init__()
        self.hidden_size = config.hidden_size
        self.FFN = LookupFFN(config, self.hidden_size)
        self.attention = Attention(config)
        self.dropout = nn.Dropout(p=config.hidden_dropout_prob)

    def _attention_and_residual(self, hidden_states, attention_mask):
        attention, dropout = self.attention, self.dropout
        if (_plain(attention, Attention) and _plain(dropout, nn.Dropout) and (not dropout.training or dropout.p == 0.0)
                and attention._kernels_apply(hidden_states, attention_mask)):
            # the residual is added where the output projection's results are stored
            return attention._forward_kernels(hidden_states, attention_mask, hidden_states)
        return dropout(attention(hidden_states, attention_mask)) + hidden_states

    def forward(self, hidden_states, attention_mask):
        attn_output = self._attention_and_residual(hidden_states, attention_mask)
        if (not self.training or self.dropout.p == 0.0) and attn_output.dtype == torch.float32:
            # dropout is the identity: the residual add runs inside the FFN's gather kernel
            return self.FFN(attn_output, residual=attn_output)
        return self.dropout(self.FFN(attn_output)) + attn_output


class Encoder(nn.Module):
    """PL/encoder.py:9-19."""

    def __init__(self, config):
        super().__init__()
        self.layer = nn.ModuleList([EncoderLayer(config) for _ in range(config.num_hidden_layers)])
        self.LayerNorm = nn.LayerNorm(config.hidden_size, eps=config.layer_norm_eps)

    def forward(self, hidden_states, attention_mask):
        for layer_module in self.layer:
            hidden_states = layer_module(hidden_states, attention_mask)
        return self.LayerNorm(hidden_states)


class Lookup(nn.Module):
    """PL/encoder.py:21-37: embeddings + encoder; returns (sequence_output, {})."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.embeddings = RobertaEmbeddings(config)
        self.encoder = Encoder(config)

    def forward(self, input_ids, token_type_ids, position_ids, attention_mask, **kwargs):
        embedding_output = self.embeddings(input_ids, token_type_ids, position_ids)
        return self.encoder(embedding_output, attention_mask), {}

    def get_input_embeddings(self):
        return self.embeddings.word_embeddings

    def set_input_embeddings(self, value):
        self.embeddings.word_embeddings = value
