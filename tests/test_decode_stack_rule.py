"""Which calls of the base model the fused decode stack takes (no GPU needed)."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from engine.kernels.paged_attention_integration import (
    DECODE_LINEAR_MAX_ROWS,
    PagedAttentionContext,
    _ids_checked,
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
