"""The reference's toy forecasting model on this engine's attention.

Reference: /root/reference src/model.py:1-92 -- PositionalEncoding,
CustomTransformerEncoderLayer (single-head SparseAttention, window 3, then a
ReLU feed-forward block, post-norm residuals) and TransformerModel
(Linear encoder * sqrt(model_dim), positional encoding, the layer stack, a
Linear decoder on the last time step).  Same class names, constructor
arguments, parameter names (so the reference's state_dicts load unchanged)
and forward semantics, including PositionalEncoding indexing its table by
``x.size(0)`` as the reference does (:19-20).  The attention inside each
layer is ``layers.SparseAttention``: the HIP kernels in eval mode, the
PyTorch path in training mode unless ``fallback_training=False``.

``fused=True`` (layer) / ``fused_layers=True`` (model), keyword-only and off
by default, runs each layer's inference forward as one HIP kernel
(ma_encoder_layer_forward, include/ma_encoder.h): attention, residual,
LayerNorm1, linear1, ReLU, linear2, residual and LayerNorm2 without
intermediate tensors.  It applies to float32 device inputs when the layer is
in eval mode (dropout the identity) and no gradient is being recorded; a call
that records gradients, or a training-mode call, runs the operations above.
A whole model of such layers, with sequences short enough for one workgroup's
LDS, runs as one launch (ma_encoder_model_forward) from the input to the
prediction; anything that would observe the modules in between (hooks,
subclasses, tracing, autocast, tensor subclasses) keeps the layer calls.
"""
from __future__ import annotations

import functools
import math

import torch
import torch.nn as nn
import torch.nn.functional as F
import torch.nn.modules.module as _module

from layers.sparse_attention import SparseAttention


class PositionalEncoding(nn.Module):
    """Sinusoidal table pe[pos, 2i] = sin(pos w_i), pe[pos, 2i+1] = cos(pos w_i),
    w_i = 10000^(-2i/d_model) (reference model.py:7-20)."""

    def __init__(self, d_model, max_len=5000):
        super().__init__()
        position = torch.arange(0, max_len, dtype=torch.float).unsqueeze(1)
        freq = torch.exp(torch.arange(0, d_model, 2).float() * (-math.log(10000.0) / d_model))
        table = torch.zeros(max_len, d_model)
        table[:, 0::2] = torch.sin(position * freq)
        table[:, 1::2] = torch.cos(position * freq)
        self.register_buffer("pe", table.unsqueeze(0).transpose(0, 1))  # [max_len, 1, d_model]

    def forward(self, x):
        return x + self.pe[:x.size(0), :]


# model widths the fused layer kernel is instantiated for (d_ff = 4 * d_model)
_FUSED_WIDTHS = (16, 32, 64, 128)


def _fused_applies(layer: nn.Module, src: torch.Tensor) -> bool:
    """Whether ``layer`` runs as the fused kernel on ``src``; otherwise it runs
    its separate operations."""
    if not (src.is_cuda and src.dtype == torch.float32) or src.dim() != 3:
        return False
    if layer.linear1.in_features not in _FUSED_WIDTHS or layer.linear1.out_features != 4 * layer.linear1.in_features:
        return False
    if layer.training and any(m.p > 0 for m in (layer.dropout, layer.dropout1, layer.dropout2)):
        return False
    if torch.is_grad_enabled() and (src.requires_grad or any(p.requires_grad for p in layer.parameters())):
        return False
    return True


def _layer_desc(layer, B: int, S: int, device):
    """The layer's ma_encoder_layer descriptor, cached on the layer per shape,
    device and parameter storage (rebuilt when any of them changes)."""
    import ma_attn as _ma
    params = (layer.norm1.weight, layer.norm1.bias, layer.linear1.weight, layer.linear1.bias,
              layer.linear2.weight, layer.linear2.bias, layer.norm2.weight, layer.norm2.bias)
    key = (B, S, device, int(layer.self_attn.window_size), layer.norm1.eps, layer.norm2.eps,
           tuple(p.data_ptr() for p in params))
    hit = getattr(layer, "_fused_desc", None)
    if hit is not None and hit[0] == key:
        return hit[1]
    if layer.norm2.eps != layer.norm1.eps:
        raise RuntimeError("the fused layer takes one LayerNorm eps for both norms")
    for p in params:
        if p.device != device or p.dtype != torch.float32 or not p.is_contiguous():
            raise RuntimeError("fused layer parameters must be contiguous float32 on the input's device")
    L = _ma.EncoderLayer()
    L.batch, L.seq_len, L.d_model = B, S, layer.linear1.in_features
    L.d_ff = layer.linear1.out_features
    L.window = int(layer.self_attn.window_size)
    L.ln_eps = float(layer.norm1.eps)
    (L.norm1_weight, L.norm1_bias, L.linear1_weight, L.linear1_bias, L.linear2_weight, L.linear2_bias,
     L.norm2_weight, L.norm2_bias) = (p.data_ptr() for p in params)
    layer._fused_desc = (key, L)
    return L


def encoder_layer_forward(layer: "CustomTransformerEncoderLayer", src: torch.Tensor,
                          attn: torch.Tensor = None) -> torch.Tensor:
    """One HIP launch for layer(src) in inference ([B, S, d_model] float32 on
    the device).  attn None: the kernel computes the layer's sliding-window
    attention too; otherwise only the block after the attention runs."""
    import ma_attn as _ma
    from sparse_attention_cuda import _on_device
    src = src.contiguous()
    B, S, Dm = src.shape
    if Dm != layer.linear1.in_features:
        raise RuntimeError(f"input width {Dm} != d_model {layer.linear1.in_features}")
    L = _layer_desc(layer, B, S, src.device)
    out = torch.empty_like(src)
    a = attn.contiguous() if attn is not None else None
    aptr = a.data_ptr() if a is not None else 0
    _on_device(src.get_device(), lambda stream: _ma.encoder_layer_forward_raw(L, src.data_ptr(), aptr,
                                                                              out.data_ptr(), stream))
    return out


class CustomTransformerEncoderLayer(nn.Module):
    """Self-attention (SparseAttention) + feed-forward, each with residual,
    dropout and post-LayerNorm (reference model.py:28-52)."""

    def __init__(self, d_model, num_heads, dropout=0.1, window_size=3, *, fallback_training=True,
                 fused=False):
        super().__init__()
        self.fused = bool(fused)
        self.self_attn = SparseAttention(window_size=window_size, fallback_training=fallback_training)
        self.linear1 = nn.Linear(d_model, d_model * 4)
        self.dropout = nn.Dropout(dropout)
        self.linear2 = nn.Linear(d_model * 4, d_model)
        self.norm1 = nn.LayerNorm(d_model)
        self.norm2 = nn.LayerNorm(d_model)
        self.dropout1 = nn.Dropout(dropout)
        self.dropout2 = nn.Dropout(dropout)

    def forward(self, src):
        if self.fused and _fused_applies(self, src):
            if self.self_attn.use_ma_core:
                return encoder_layer_forward(self, src)
            # the layer's own PyTorch attention (a different mask), then the fused block
            return encoder_layer_forward(self, src, self.self_attn(src, src, src))
        attn = self.self_attn(src, src, src)
        src = self.norm1(src + self.dropout1(attn))
        ff = self.linear2(self.dropout(F.relu(self.linear1(src))))
        return self.norm2(src + self.dropout2(ff))


def _plain(module: nn.Module, cls) -> bool:
    """Whether calling `module` runs cls.forward and nothing else."""
    return (type(module) is cls and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks))


@functools.lru_cache(maxsize=16)
def _model_shapes(D: int, inputs: int, layers: int) -> list:
    block = [(D,), (D,), (4 * D, D), (4 * D,), (D, 4 * D), (D,), (D,), (D,)]
    return [(D, inputs), (D,), (1, D), (1,)] + block * layers


def _model_params(model: "TransformerModel"):
    """The parameters encoder_model_forward reads (encoder, decoder, then each
    layer's norm1, linear1, linear2, norm2; weight before bias) and the layers'
    (window, eps), or None when the model holds anything but plain modules of
    the shapes its constructor gives them: a replaced head, for instance."""
    mods = model._modules
    enc, pos, dec, layers = mods["encoder"], mods["pos_encoder"], mods["decoder"], mods["encoder_layers"]
    D = model.model_dim
    if D not in _FUSED_WIDTHS or not (_plain(enc, nn.Linear) and _plain(dec, nn.Linear)
                                      and _plain(pos, PositionalEncoding)):
        return None
    pairs, windows = [enc._parameters, dec._parameters], []
    for layer in layers._modules.values():
        if not (_plain(layer, CustomTransformerEncoderLayer) and layer.fused):
            return None
        sub = layer._modules
        attn, n1, n2 = sub["self_attn"], sub["norm1"], sub["norm2"]
        if not (type(attn) is SparseAttention and attn.use_ma_core) or n1.eps != n2.eps:
            return None
        if layer.training and any(sub[n].p > 0 for n in ("dropout", "dropout1", "dropout2")):
            return None
        pairs += (n1._parameters, sub["linear1"]._parameters, sub["linear2"]._parameters, n2._parameters)
        windows.append((int(attn.window_size), float(n1.eps)))
    params = [p.get(n) for p in pairs for n in ("weight", "bias")]
    shapes = [None if p is None else p.shape for p in params]
    return (params, windows) if shapes == _model_shapes(D, enc.in_features, len(windows)) else None


def _observed() -> bool:
    """Whether something would see the operations inside a call: global hooks,
    autocast, tracing, torch modes or function transforms.  A torch that lacks
    one of the (partly private) names asked here counts as observing."""
    try:
        return bool(_module._global_forward_hooks or _module._global_forward_pre_hooks
                    or torch.is_autocast_enabled("cuda") or torch.jit.is_tracing() or torch.compiler.is_compiling()
                    or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                    or torch._C._functorch.peek_interpreter_stack() is not None)
    except (AttributeError, TypeError):
        return True


def _model_launch(model: "TransformerModel", src: torch.Tensor):
    """model(src) as one launch, or None when the call needs its modules:
    gradients, training-mode dropout, other types, hooks, a width, depth,
    length or parameter shape the kernel does not take."""
    if type(src) is not torch.Tensor or not src.is_cuda or src.dtype != torch.float32 or src.dim() != 3 or \
            _observed():
        return None
    B, S, I = src.shape
    found = _model_params(model) if B > 0 and S > 0 else None
    if found is None:
        return None
    params, windows = found
    D, pe, dev = model.model_dim, model._modules["pos_encoder"]._buffers["pe"], src.device
    if pe.dtype != torch.float32 or pe.device != dev or pe.shape[0] < B or pe.shape[1:] != (1, D) or \
            not pe.is_contiguous() or pe.data_ptr() % 16:
        return None
    grad = torch.is_grad_enabled()
    ptrs, low = [], 0
    for p in params:
        if p.device != dev or p.dtype != torch.float32 or not p.is_contiguous() or (grad and p.requires_grad):
            return None
        ptrs.append(p.data_ptr())
        low |= ptrs[-1]
    if (grad and src.requires_grad) or params[0].shape[1] != I:
        return None
    if low % 16 and any(p % 16 for p in ptrs[1:3] + ptrs[4:]):  # encoder.weight and decoder.bias may lie anywhere
        return None
    import ma_attn as _ma
    if len(windows) < 1 or len(windows) > _ma.ENCODER_MAX_LAYERS or S > _ma.LIB.ma_encoder_model_max_seq(D):
        return None
    from sparse_attention_cuda import _on_device
    descs = (_ma.EncoderLayer * len(windows))()
    for i, (w, eps) in enumerate(windows):
        descs[i] = _ma.EncoderLayer(B, S, D, 4 * D, w, eps, 0, *ptrs[4 + 8 * i:12 + 8 * i])
    M = _ma.EncoderModel(B, S, I, D, len(windows), descs, ptrs[0], ptrs[1], pe.data_ptr(), ptrs[2], ptrs[3])
    src = src.contiguous()
    out = torch.empty((B, 1), dtype=torch.float32, device=src.device)
    _on_device(src.get_device(),
               lambda stream: _ma.encoder_model_forward_raw(M, src.data_ptr(), out.data_ptr(), stream))
    return out


class TransformerModel(nn.Module):
    """[batch, seq_len, input_dim] -> [batch, 1] (reference model.py:54-92).

    num_heads is accepted and unused, as in the reference (its layers are
    single-head)."""

    def __init__(self, input_dim, model_dim, num_heads, num_layers, dropout=0.1, *,
                 fallback_training=True, fused_layers=False):
        super().__init__()
        self.model_dim = model_dim
        self.fused_layers = bool(fused_layers)
        self.encoder = nn.Linear(input_dim, model_dim)
        self.pos_encoder = PositionalEncoding(model_dim)
        self.encoder_layers = nn.ModuleList([
            CustomTransformerEncoderLayer(d_model=model_dim, num_heads=num_heads, dropout=dropout,
                                          fallback_training=fallback_training, fused=fused_layers)
            for _ in range(num_layers)
        ])
        self.decoder = nn.Linear(model_dim, 1)
        self.init_weights()

    def init_weights(self):
        r = 0.1
        self.encoder.weight.data.uniform_(-r, r)
        self.decoder.bias.data.zero_()
        self.decoder.weight.data.uniform_(-r, r)

    def forward(self, src):
        if self.__dict__.get("fused_layers"):  # absent from models pickled before it existed
            out = _model_launch(self, src)
            if out is not None:
                return out
        x = self.pos_encoder(self.encoder(src) * math.sqrt(self.model_dim))
        for layer in self.encoder_layers:
            x = layer(x)
        return self.decoder(x[:, -1, :])
