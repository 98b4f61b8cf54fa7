"""The decoder model with parts that are not its own: whatever stands in a
layer's or an attention's place is called with rows, residual, metadata, cache
and angles (an attention without the residual), as the model's own modules can
be, and nothing else is asked of it."""

import pytest
import torch
from torch import nn

from fusioninfer_amd.config import CacheConfig, EngineConfig, SchedulerConfig
from fusioninfer_amd.engine.llm_engine import LLMEngine
from fusioninfer_amd.engine.sequence import SamplingParams
from fusioninfer_amd.models.model import DecoderLayer
from fusioninfer_amd.models.registry import get_model_config

PROMPT = [3, 1, 4, 1, 5, 9, 2, 6, 5]


def make_engine(name="tiny-qwen3", layers=3, quantization=None):
    mc = get_model_config(name)
    mc.num_layers = layers
    mc.quantization = quantization
    return LLMEngine(EngineConfig(
        model=mc, cache=CacheConfig(num_gpu_blocks=64),
        scheduler=SchedulerConfig(max_num_seqs=4, max_num_batched_tokens=256,
                                  max_model_len=128)), device="cpu")


def states(eng, caches=None):
    """Of all rows, from the model itself; of the first caches' layers."""
    seen = []
    forward = type(eng.runner.model).forward

    class Seen(type(eng.runner.model)):
        def forward(self, ids, meta, kv_caches):
            seen.append(forward(self, ids, meta, kv_caches[:caches]))
            return seen[-1]

    model, eng.runner.model.__class__ = type(eng.runner.model), Seen
    try:
        eng.embed([PROMPT])
    finally:
        eng.runner.model.__class__ = model
    return seen[0]


class Inside(nn.Module):
    """Calls the layer, or the attention, in whose place it stands."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner
        self.calls = 0

    def forward(self, *args):
        self.calls += 1
        return self.inner(*args)


class LayerInside(Inside):
    def forward(self, hidden, residual, meta, kv_cache, cos_sin):
        return super().forward(hidden, residual, meta, kv_cache, cos_sin)


CONFIGS = [("tiny-qwen3", None), ("tiny-qwen3", "fp8"),
           ("tiny-qwen3-moe", None)]


@pytest.mark.parametrize("name,quantization", CONFIGS)
@pytest.mark.parametrize("places", [[0], [1], [2], [0, 1, 2]])
def test_module_in_a_layers_place(name, quantization, places):
    eng = make_engine(name, quantization=quantization)
    want = states(eng)
    layers = eng.runner.model.layers
    for i in places:
        layers[i] = LayerInside(layers[i])
    assert torch.equal(states(eng), want)
    assert all(layers[i].calls == 1 for i in places)


class AttentionInside(Inside):
    def forward(self, x, meta, kv_cache, cos_sin):
        return super().forward(x, meta, kv_cache, cos_sin)


@pytest.mark.parametrize("name,quantization", CONFIGS)
@pytest.mark.parametrize("places", [[0], [1, 2]])
def test_module_in_an_attentions_place(name, quantization, places):
    eng = make_engine(name, quantization=quantization)
    want = states(eng)
    layers = eng.runner.model.layers
    for i in places:
        layers[i].self_attn = AttentionInside(layers[i].self_attn)
    assert torch.equal(states(eng), want)
    assert all(layers[i].self_attn.calls == 1 for i in places)


@pytest.mark.parametrize("name,quantization", CONFIGS)
@pytest.mark.parametrize("caches", [1, 2])
def test_state_after_the_first_layers(name, quantization, caches):
    """The caches say how many layers run, and the last norm is behind the
    last of these: as in a model whose other layers are not there."""
    eng = make_engine(name, quantization=quantization)
    got = states(eng, caches)
    eng.runner.model.layers = eng.runner.model.layers[:caches]
    assert torch.equal(got, states(eng))


def test_models_forward_as_ever():
    """A forward without the rows to give, of a class of its own or set on the
    model, serves; whoever hooks the model sees the state of all rows."""
    eng = make_engine()
    model = eng.runner.model
    cls = type(model)
    seen = []

    def tokens():
        return eng.generate([PROMPT], SamplingParams(max_tokens=3))[0] \
            .output_token_ids

    def forward(self, ids, meta, kv_caches):
        seen.append(cls.forward(self, ids, meta, kv_caches).shape)
        return cls.forward(self, ids, meta, kv_caches)

    want = tokens()
    model.__class__ = type("Own", (cls,), {"forward": forward})
    assert tokens() == want
    model.__class__ = cls
    model.forward = lambda *args: forward(model, *args)
    assert tokens() == want
    del model.forward
    hook = model.register_forward_hook(
        lambda _, args, out: seen.append(out.shape))
    assert tokens() == want
    hook.remove()
    width = model.cfg.hidden_size
    assert seen == 3 * [(len(PROMPT), width), (1, width), (1, width)]


@pytest.mark.parametrize("stream", [False, True])
def test_no_row_wanted(stream, monkeypatch):
    """Nothing, in the model's type, of a stream that is kept in fp32 too."""
    eng = make_engine()
    model = eng.runner.model
    if stream:
        monkeypatch.setattr(
            DecoderLayer, "forward",
            lambda self, hidden, residual, *_, **__: (None, (
                hidden if residual is None else residual).float()))
    else:
        monkeypatch.setattr(
            DecoderLayer, "forward",
            lambda self, hidden, residual, *_, **__: (hidden, hidden))
    got = model(torch.tensor(PROMPT), None, eng.runner.kv_caches,
                rows=torch.empty(0, dtype=torch.long))
    assert got.shape == (0, model.cfg.hidden_size)
    assert got.dtype == torch.bfloat16
