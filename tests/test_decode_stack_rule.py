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
    _stack_layer,
    _stack_sizes,
    _stack_takes,
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


def _packed_layer():
    """A decoder layer with the sizes that the packed copies leave on it (no copies needed here)."""
    from transformers import Qwen2Config
    from transformers.models.qwen2.modeling_qwen2 import Qwen2DecoderLayer

    layer = Qwen2DecoderLayer(Qwen2Config(hidden_size=64, intermediate_size=96,
                                          num_attention_heads=2, num_key_value_heads=1,
                                          head_dim=16), 0).half()
    layer._pa_packed = (torch.zeros(1, dtype=torch.float16),) * 4
    layer._pa_sizes = _stack_sizes(layer)
    return layer


def test_weights_the_kernels_cannot_read_take_the_layers():
    """The parameters that the stack reads in place: another type, shape, stride or alignment."""
    half = dict(dtype=torch.float16)
    good = _stack_layer(_packed_layer(), 3)
    assert good.o.shape == (64, 32) and (good.q_width, good.kv_width) == (32, 16)

    def replaced(module, weight, name="weight"):
        layer = _packed_layer()
        owner = layer.get_submodule(module)
        setattr(owner, name, torch.nn.Parameter(weight, requires_grad=False))
        return _stack_layer(layer, 3)

    o, down, norm = "self_attn.o_proj", "mlp.down_proj", "input_layernorm"
    wide, odd = torch.zeros(64, 40, **half), torch.zeros(64 * 32 + 4, **half)
    assert replaced(o, wide[:, :32]).o.stride() == (40, 1)
    assert replaced(o, torch.zeros(64, **half), "bias").o_bias is not None
    for module, weight in ((o, torch.zeros(64, 32)), (o, torch.zeros(64, 64, **half)),
                           (o, torch.zeros(32, 64, **half).t()),
                           (o, torch.zeros(64, 36, **half)[:, :32]), (o, odd[4:].view(64, 32)),
                           (down, torch.zeros(64, 64, **half)), (norm, torch.zeros(64)),
                           (norm, torch.zeros(65, **half)[1:]), (norm, torch.zeros(128, **half)[::2])):
        assert replaced(module, weight) is None
    assert replaced(o, torch.zeros(64), "bias") is None
    layer = _packed_layer()
    torch.nn.utils.parametrize.register_parametrization(layer.mlp.down_proj, "weight",
                                                        torch.nn.Identity())
    assert _stack_layer(layer, 3) is None


def _layer(hidden, mlp, heads, kv_heads, dim):
    """A layer of these sizes without storage."""
    weight = lambda n, k: SimpleNamespace(  # noqa: E731
        weight=torch.empty(n, k, dtype=torch.float16, device="meta"))
    return SimpleNamespace(
        self_attn=SimpleNamespace(q_proj=weight(heads * dim, hidden),
                                  k_proj=weight(kv_heads * dim, hidden)),
        mlp=SimpleNamespace(down_proj=weight(hidden, mlp)))


# The sizes measured beside DECODE_LINEAR_ROWS: up to the last row count at which the stack was not
# the slower path, or fewer.
@pytest.mark.parametrize("sizes,rows", [
    ((896, 4864, 14, 2, 64), 256), ((1536, 8960, 12, 2, 128), 128), ((2048, 5504, 16, 16, 128), 128),
    ((2048, 11008, 16, 2, 128), 128), ((2560, 9728, 32, 8, 128), 128),
    ((4096, 11008, 32, 32, 128), 64), ((3584, 18944, 28, 4, 128), 64),
    ((5120, 27648, 40, 8, 128), 64), ((8192, 29568, 64, 8, 128), 32)])
def test_rows_by_layer_size(sizes, rows):
    assert _stack_sizes(_layer(*sizes)).rows == rows


def test_more_rows_than_the_layers_size_allows_take_the_layers(monkeypatch):
    from transformers import Qwen2Config
    from transformers.models.qwen2.modeling_qwen2 import Qwen2Model

    m = Qwen2Model(Qwen2Config(vocab_size=32, hidden_size=64, intermediate_size=96,
                               num_hidden_layers=2, num_attention_heads=2, num_key_value_heads=1))
    m._paged_stack_context = SimpleNamespace(is_decode=True, is_batched=True)
    m._orig_stack_forward = lambda **kwargs: "layers"
    for i in range(2):
        m.layers[i] = _packed_layer()
    m.layers[1]._pa_sizes = m.layers[1]._pa_sizes._replace(rows=16)
    monkeypatch.setattr(integration, "_plain_embedding_and_rope", lambda m: 1 / 0)  # the stack itself

    def call(rows):
        ids = torch.zeros(rows, 1, dtype=torch.long)
        return integration.fused_decoder_stack_forward(m, input_ids=ids, position_ids=ids,
                                                       use_cache=False)

    assert call(17) == "layers"
    with pytest.raises(ZeroDivisionError):
        call(16)
