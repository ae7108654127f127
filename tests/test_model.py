"""The toy TransformerModel (reference src/model.py) on the engine's attention:
structure and CPU semantics (no GPU needed)."""
import math

import pytest
import torch
import torch.nn.functional as F


def _window_attention(x, w):
    """Single-head attention over keys |i - j| <= w, written with torch SDPA."""
    S, D = x.shape[1], x.shape[2]
    i = torch.arange(S)
    mask = (i.view(-1, 1) - i.view(1, -1)).abs() <= w
    return F.scaled_dot_product_attention(x.unsqueeze(1), x.unsqueeze(1), x.unsqueeze(1), attn_mask=mask,
                                          scale=1.0 / math.sqrt(D)).squeeze(1)


def _manual_forward(m, src):
    """The reference forward (model.py:80-91, :42-52) restated with SDPA."""
    x = m.encoder(src) * math.sqrt(m.model_dim)
    x = x + m.pos_encoder.pe[:x.size(0), :]
    for layer in m.encoder_layers:
        x = layer.norm1(x + _window_attention(x, layer.self_attn.window_size))
        x = layer.norm2(x + layer.linear2(F.relu(layer.linear1(x))))
    return m.decoder(x[:, -1, :])


def test_state_dict_names_match_reference():
    from model import TransformerModel
    m = TransformerModel(input_dim=5, model_dim=32, num_heads=2, num_layers=2)
    want = {"encoder.weight", "encoder.bias", "pos_encoder.pe", "decoder.weight", "decoder.bias"}
    for l in range(2):
        for n in ("linear1", "linear2", "norm1", "norm2"):
            want |= {f"encoder_layers.{l}.{n}.weight", f"encoder_layers.{l}.{n}.bias"}
    assert set(m.state_dict()) == want
    assert m.pos_encoder.pe.shape == (5000, 1, 32)


@pytest.mark.parametrize("model_dim,num_layers", [(32, 2), (64, 4)])
def test_cpu_forward_matches_restatement(model_dim, num_layers):
    from model import TransformerModel
    torch.manual_seed(0)
    m = TransformerModel(input_dim=5, model_dim=model_dim, num_heads=2, num_layers=num_layers).eval()
    src = torch.randn(64, 10, 5)
    with torch.no_grad():
        out = m(src)
        ref = _manual_forward(m, src)
    assert out.shape == (64, 1)
    torch.testing.assert_close(out, ref, rtol=1e-5, atol=1e-5)


def _grown(lin):
    lin.weight = torch.nn.Parameter(torch.zeros(lin.weight.shape[0], lin.weight.shape[1] + 1))


@pytest.mark.parametrize("change", [
    lambda m: setattr(m, "decoder", torch.nn.Linear(32, 3)),
    lambda m: setattr(m, "decoder", torch.nn.Linear(16, 1)),
    lambda m: setattr(m, "decoder", torch.nn.Linear(32, 1, bias=False)),
    lambda m: setattr(m, "encoder", torch.nn.Linear(5, 16)),
    lambda m: setattr(m.encoder_layers[1], "linear2", torch.nn.Linear(64, 32)),
    lambda m: setattr(m.encoder_layers[1], "linear1", torch.nn.Linear(32, 64)),
    lambda m: setattr(m.encoder_layers[0], "norm2", torch.nn.LayerNorm(16)),
    lambda m: setattr(m.encoder_layers[0], "norm1", torch.nn.LayerNorm((1, 32))),
    lambda m: _grown(m.encoder),
    lambda m: _grown(m.encoder_layers[0].linear2),
], ids=["head3", "head16", "no_bias", "encoder16", "linear2", "linear1", "norm2", "norm1_2d", "encoder_in", "ff_in"])
def test_one_launch_needs_the_constructors_shapes(change):
    """The one-launch model takes pointers only, so a model whose modules were
    replaced by ones of other shapes keeps its modules' own forward."""
    from model import TransformerModel, _model_params
    m = TransformerModel(input_dim=5, model_dim=32, num_heads=2, num_layers=2, fused_layers=True).eval()
    params, windows = _model_params(m)
    assert len(params) == 4 + 8 * 2 and windows == [(3, 1e-5)] * 2
    src = torch.randn(3, 10, 5)
    with torch.no_grad():
        assert m(src).shape == (3, 1)
        change(m)
        if m.decoder.out_features == 3:
            assert m(src).shape == (3, 3)
    found = _model_params(m)  # the encoder's input width is compared with the call's
    assert found is None or found[0][0].shape[1] != src.shape[2]


@pytest.mark.parametrize("where,name", [(torch._C, "_len_torch_dispatch_stack"), (torch._C, "_len_torch_function_stack"),
                                        (torch._C._functorch, "peek_interpreter_stack"),
                                        (torch.nn.modules.module, "_global_forward_pre_hooks")])
def test_one_launch_stays_off_without_a_private_name(monkeypatch, where, name):
    """The one-launch model asks torch, partly by private names, whether
    anything observes the call; a torch without one of them keeps the modules."""
    from model import _observed
    assert _observed() is False
    monkeypatch.delattr(where, name)
    assert _observed() is True
