"""Which calls of the base model the fused decode stack takes (no GPU needed)."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from engine.kernels import paged_attention_integration as integration
from engine.kernels.paged_attention_integration import (
    DECODE_LINEAR_MAX_ROWS,
    PagedAttentionContext,
    _ids_checked,
    _max_rows,
    _stack_takes,
    _weights_readable,
)


@pytest.fixture(scope="module")
def model():
    from transformers import Qwen2Config
    from transformers.models.qwen2.modeling_qwen2 import Qwen2Model

    m = Qwen2Model(Qwen2Config(vocab_size=32, hidden_size=32, intermediate_size=32,
                               num_hidden_layers=2, num_attention_heads=2, num_key_value_heads=1))
    m._paged_stack_context = SimpleNamespace(is_decode=True, is_batched=True)
    return m


def _takes(model, rows=3, width=1, mask=None, positions=True, cache=None, embeds=None,
           use_cache=False, **kwargs):
    ids = torch.zeros(rows, width, dtype=torch.long)
    return _stack_takes(model, ids, mask, torch.zeros(rows, 1) if positions else None, cache,
                        embeds, use_cache, kwargs)


def test_plain_decode_steps_are_taken(model):
    assert _takes(model) and _takes(model, rows=DECODE_LINEAR_MAX_ROWS)
    assert _takes(model, output_hidden_states=False, cache_position=None)


@pytest.mark.parametrize("call", [
    dict(rows=DECODE_LINEAR_MAX_ROWS + 1), dict(rows=0), dict(width=2), dict(mask=torch.ones(3, 1)),
    dict(positions=False), dict(cache=object()), dict(embeds=torch.zeros(3, 1, 32)),
    dict(use_cache=True), dict(output_hidden_states=True), dict(output_attentions=True),
    dict(return_dict=False), dict(use_cache=None), dict(cache_position=torch.arange(3)), dict(cache_position=torch.zeros(1)),
])
def test_calls_that_ask_for_more_take_the_layers(model, call):
    assert not _takes(model, **call)


def test_hooks_and_contexts_take_the_layers(model):
    for register in (model.layers[1].register_forward_hook,
                     model.layers[0].register_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not _takes(model)
        handle.remove()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not _takes(model)
    handle.remove()
    for context in (None, SimpleNamespace(is_decode=False, is_batched=True),
                    SimpleNamespace(is_decode=True, is_batched=False)):
        own, model._paged_stack_context = model._paged_stack_context, context
        assert not _takes(model)
        model._paged_stack_context = own
    model.config.output_hidden_states = True
    assert not _takes(model)
    model.config.output_hidden_states = False
    assert _takes(model)


@pytest.mark.parametrize("config", [{}, {"use_cache": False}, {"return_dict": False}])
@pytest.mark.parametrize("call", [
    {}, {"use_cache": None}, {"use_cache": False}, {"use_cache": False, "return_dict": None},
    {"use_cache": False, "return_dict": True}, {"use_cache": False, "return_dict": False}])
def test_calls_taken_return_hidden_states_alone(config, call):
    """What the replaced forward returns, wherever the stack takes its call: a model output that
    holds the last hidden states and nothing else."""
    from transformers import Qwen2Config
    from transformers.modeling_outputs import BaseModelOutputWithPast
    from transformers.models.qwen2.modeling_qwen2 import Qwen2Model

    m = Qwen2Model(Qwen2Config(vocab_size=32, hidden_size=32, intermediate_size=32,
                               num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=1,
                               **config))
    m._paged_stack_context = SimpleNamespace(is_decode=True, is_batched=True)
    ids, pos = torch.zeros(3, 1, dtype=torch.long), torch.zeros(3, 1, dtype=torch.long)
    out = m(input_ids=ids, position_ids=pos, **call)
    alone = isinstance(out, BaseModelOutputWithPast) and list(out.keys()) == ["last_hidden_state"]
    kwargs = {k: v for k, v in call.items() if k != "use_cache"}
    assert _stack_takes(m, ids, None, pos, None, None, call.get("use_cache"), kwargs) == alone


def test_only_ids_checked_against_the_table_skip_the_embedding_module():
    emb = torch.nn.Embedding(8, 4)
    pool = SimpleNamespace(device=torch.device("cpu"))
    ctx = PagedAttentionContext.from_device(pool, None, None)
    assert not _ids_checked(ctx, emb) and not _ids_checked(SimpleNamespace(), emb)
    for checked, taken in ((8, True), (5, True), (9, False)):
        ctx.checked_vocab = checked
        assert _ids_checked(ctx, emb) == taken


def test_weights_the_kernels_cannot_read_take_the_layers():
    """The parameters that the stack reads in place: another type, shape, stride or alignment."""
    half = dict(dtype=torch.float16)

    def layer():
        linear = lambda n, k: SimpleNamespace(weight=torch.zeros(n, k, **half), bias=None,  # noqa: E731
                                              out_features=n)
        norm = lambda: SimpleNamespace(weight=torch.zeros(64, **half))  # noqa: E731
        return SimpleNamespace(
            self_attn=SimpleNamespace(o_proj=linear(64, 32), q_proj=linear(32, 64)),
            mlp=SimpleNamespace(down_proj=linear(64, 96)), input_layernorm=norm(),
            post_attention_layernorm=norm(),
            _pa_packed=(torch.zeros(4, 2, 4, 16, 8, **half), torch.zeros(12, 2, 4, 16, 8, **half)))

    assert _weights_readable(layer())
    wide, odd = torch.zeros(64, 40, **half), torch.zeros(64 * 32 + 4, **half)
    m = layer()
    m.self_attn.o_proj.weight = wide[:, :32]
    assert _weights_readable(m)
    for name, weight in (("o_proj", torch.zeros(64, 32)), ("o_proj", torch.zeros(64, 64, **half)),
                         ("o_proj", torch.zeros(32, 64, **half).t()),
                         ("o_proj", torch.zeros(64, 36, **half)[:, :32]),
                         ("o_proj", odd[4:].view(64, 32)),
                         ("down_proj", torch.zeros(64, 64, **half))):
        m = layer()
        getattr(m.self_attn if name == "o_proj" else m.mlp, name).weight = weight
        assert not _weights_readable(m)
    m = layer()
    m.self_attn.o_proj.bias = torch.zeros(64)
    assert not _weights_readable(m)
    m = layer()
    m.input_layernorm.weight = torch.zeros(65, **half)[1:]
    assert not _weights_readable(m)


def _layer(hidden, mlp, heads, kv_heads, dim):
    """A prepared layer of these sizes without storage."""
    empty = lambda *shape: torch.empty(shape, dtype=torch.float16, device="meta")  # noqa: E731
    qkv = (heads + 2 * kv_heads) * dim
    return SimpleNamespace(
        self_attn=SimpleNamespace(o_proj=SimpleNamespace(weight=empty(hidden, heads * dim))),
        mlp=SimpleNamespace(down_proj=SimpleNamespace(weight=empty(hidden, mlp))),
        _pa_packed=(empty(qkv // 16, hidden // 32, 4, 16, 8),
                    empty(2 * mlp // 16, hidden // 32, 4, 16, 8)))


# The sizes measured beside DECODE_LINEAR_ROWS: up to the last row count at which the stack was not
# the slower path, or fewer.
@pytest.mark.parametrize("sizes,rows", [
    ((896, 4864, 14, 2, 64), 256), ((1536, 8960, 12, 2, 128), 128), ((2048, 5504, 16, 16, 128), 128),
    ((2048, 11008, 16, 2, 128), 128), ((2560, 9728, 32, 8, 128), 128),
    ((4096, 11008, 32, 32, 128), 64), ((3584, 18944, 28, 4, 128), 64),
    ((5120, 27648, 40, 8, 128), 64), ((8192, 29568, 64, 8, 128), 32)])
def test_rows_by_layer_size(sizes, rows):
    assert _max_rows(_layer(*sizes)) == rows


def test_more_rows_than_the_layers_size_allows_take_the_layers(model, monkeypatch):
    monkeypatch.setattr(model, "_orig_stack_forward", lambda **kwargs: "layers", raising=False)
    monkeypatch.setattr(integration, "_weights_readable", lambda layer: True)
    monkeypatch.setattr(integration, "_max_rows", lambda layer: 16 if layer is model.layers[1] else 64)
    monkeypatch.setattr(integration, "_plain_embedding_and_rope", lambda m: 1 / 0)  # the stack itself

    def call(rows):
        ids = torch.zeros(rows, 1, dtype=torch.long)
        return integration.fused_decoder_stack_forward(model, input_ids=ids, position_ids=ids,
                                                       use_cache=False)

    assert call(17) == "layers"
    with pytest.raises(ZeroDivisionError):
        call(16)
