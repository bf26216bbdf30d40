"""Host side of the MoE layer's calls: what a call hands to the library and
what it leaves behind, with a stand-in for the library (no device)."""
import types

import pytest


@pytest.fixture
def layer():
    import torch
    from vates_amd.moe import MoELayer, QuantizedProj

    def stack(n, rows, cols, bits=4):
        z = torch.zeros((n, rows, cols // 64), dtype=torch.int16)
        return QuantizedProj(torch.zeros((n, rows, cols * bits // 32), dtype=torch.int32), z, z.clone())

    return MoELayer(stack(1, 64, 512, 8), stack(64, 64, 512), stack(64, 64, 512), stack(64, 512, 64), top_k=4)


def test_prefill_without_tables_leaves_the_descriptor_alone(layer, monkeypatch):
    """Two prefill(use_tables=False) calls that overlap (the second runs inside
    the first's library call, as another thread's may): the library gets
    descriptors without tables, and the layer's own keeps them throughout."""
    import torch
    from vates_amd import moe
    tables = torch.zeros(16, dtype=torch.uint8)
    layer._pf_tables = tables
    layer.desc.prefill_tables = tables.data_ptr()
    x, ws = torch.zeros((2, 512), dtype=torch.bfloat16), torch.zeros(16, dtype=torch.uint8)
    stream = types.SimpleNamespace(cuda_stream=0)
    seen = []

    def vmi_moe_prefill(desc, *args):
        seen.append((desc._obj.prefill_tables, layer.desc.prefill_tables))
        if len(seen) == 1:
            layer.prefill(x, use_tables=False, stream=stream, ws=ws)
            seen.append((desc._obj.prefill_tables, layer.desc.prefill_tables))
        return 0

    monkeypatch.setattr(moe, "load", lambda: types.SimpleNamespace(vmi_moe_prefill=vmi_moe_prefill))
    layer.prefill(x, use_tables=False, stream=stream, ws=ws)
    assert seen == [(None, tables.data_ptr())] * 3
    assert layer.desc.prefill_tables == tables.data_ptr()
