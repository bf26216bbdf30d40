"""Which prompts decode.prefill may take through the prompt kernels: only models
whose layers run this package's own forward (no device: stand-in layers whose
prompt forms are all supported)."""
import types

import pytest
import torch


def _layer(cls, **kw):
    obj = cls.__new__(cls)
    obj.__dict__.update(kw)
    return obj


def _model(cls=None):
    from vates_amd.attention import AttentionLayer, KVCache
    from vates_amd.decode import DecoderLayer, SpecModel
    from vates_amd.gdn import GatedDeltaNetLayer, GdnCache
    from vates_amd.moe import MoELayer
    moe, attn, gdn = (_layer(c) for c in (MoELayer, AttentionLayer, GatedDeltaNetLayer))
    attn.__dict__.update(n_heads=4, n_kv=2)
    model = _layer(cls or SpecModel, layers=[DecoderLayer(moe, gdn=gdn), DecoderLayer(moe, attn=attn)])
    return model, [_layer(GdnCache, n_slots=9), _layer(KVCache, max_len=64)]


@pytest.fixture(autouse=True)
def supported(monkeypatch):
    from vates_amd.attention import AttentionLayer
    from vates_amd.gdn import GatedDeltaNetLayer
    from vates_amd.moe import MoELayer
    from vates_amd.mtp import MTPLayer
    for cls in (MoELayer, AttentionLayer, GatedDeltaNetLayer):
        monkeypatch.setattr(cls, "prompt_workspace_bytes", lambda self, T: 256)
    monkeypatch.setattr(MTPLayer, "fill_workspace_bytes", lambda self, T: 256)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def _blocks(model, caches, drafter=None):
    from vates_amd.decode import _prompt_blocks
    return _prompt_blocks(model, torch.zeros(40, dtype=torch.int32), caches, drafter, 8)


def test_own_layers_take_the_prompt_kernels():
    assert _blocks(*_model()) == [(0, 40)]


def test_other_layers_keep_their_own_forward():
    from vates_amd.decode import SpecModel
    from vates_amd.moe import MoELayer
    from vates_amd.mtp import MTPLayer

    class Wrapped:  # any callable served as a decoder layer's MoE
        def __init__(self, moe):
            self.moe = moe

        def __call__(self, *args, **kw):
            return self.moe(*args, **kw)

    class Counting(MoELayer):
        def __call__(self, *args, **kw):
            return super().__call__(*args, **kw)

    class Tapped(SpecModel):
        def forward(self, *args, **kw):
            return super().forward(*args, **kw)

    model, caches = _model()
    model.layers[0].moe = Wrapped(model.layers[0].moe)
    assert _blocks(model, caches) == []
    model, caches = _model()
    model.layers[1].moe = _layer(Counting)
    assert _blocks(model, caches) == []
    assert _blocks(*_model(Tapped)) == []
    model, caches = _model()
    model.forward = lambda *args, **kw: SpecModel.forward(model, *args, **kw)
    assert _blocks(model, caches) == []
    # an MTP layer's forward
    model, caches = _model()
    mtp = _layer(MTPLayer, w=types.SimpleNamespace(attn=model.layers[1].attn))
    drafter = types.SimpleNamespace(mtp=mtp, cache=caches[1])
    assert _blocks(model, caches, drafter) == [(0, 40)]
    mtp.advance = lambda *args, **kw: None
    assert _blocks(model, caches, drafter) == []


def test_blocks_halve_where_the_workspace_does_not_fit(monkeypatch):
    from vates_amd import decode
    model, caches = _model()
    prompt = torch.zeros(100, dtype=torch.int32)
    asked, room = [], 0

    def scratch(nbytes, device, stream=None):
        asked.append(nbytes)
        if nbytes > room:
            raise torch.OutOfMemoryError("stand-in")
        return nbytes

    monkeypatch.setattr(type(model.layers[0].moe), "prompt_workspace_bytes", lambda self, T: 10 * T)
    monkeypatch.setattr(decode, "scratch", scratch)
    room = 300
    assert decode._prompt_scratch(model, prompt, [(0, 100)], None) == ([(0, 25), (25, 50), (50, 75), (75, 100)], 256)
    room = 200  # 13 tokens: no prompt block any more
    assert decode._prompt_scratch(model, prompt, [(0, 100)], None) == ([], None)
    assert asked == [1000, 500, 256, 1000, 500, 256]


def test_prompt_entries_refuse_other_shapes():
    """A shape that the kernels' grids do not fit is refused before the library is called."""
    from vates_amd._lib import VmiError
    from vates_amd.attention import qgemm
    from vates_amd.moe import QuantizedProj
    model, (gdn_cache, kv_cache) = _model()
    bf16 = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)  # noqa: E731
    for layer in model.layers:
        for part in (layer.moe, layer.attn, layer.gdn):
            if part is not None:
                part.__dict__.update(hidden=512, device=torch.device("cpu"))
    gdn, attn = model.layers[0].gdn, model.layers[1].attn
    gdn.__dict__.update(n_k=2, n_v=4)
    gdn_cache.__dict__.update(n_k=2, n_v=4)
    kv_cache.n_kv = 2
    w = QuantizedProj(torch.zeros((1, 16, 64), dtype=torch.int32), bf16(1, 16, 8), bf16(1, 16, 8))
    for call in (lambda: model.layers[0].moe.prompt(bf16(20, 1024)), lambda: model.layers[0].moe.prompt(bf16(512)),
                 lambda: attn.prompt(bf16(20, 1024), kv_cache, pos0=0), lambda: gdn.prompt(bf16(20, 256), gdn_cache, pos0=0),
                 lambda: qgemm(bf16(20, 1024), w, bf16(20, 16)), lambda: qgemm(bf16(20, 512), w, bf16(20, 8))):
        with pytest.raises(VmiError):
            call()
    kv_cache.n_kv, gdn_cache.n_v = 1, 2
    for call in (lambda: attn.prompt(bf16(20, 512), kv_cache, pos0=0), lambda: gdn.prompt(bf16(20, 512), gdn_cache, pos0=0)):
        with pytest.raises(VmiError):
            call()
