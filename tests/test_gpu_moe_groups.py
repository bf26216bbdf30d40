"""GPU tests of the MoE layer on batches of more than eight tokens, which
k_route deals into token groups per slot: every row, id and score equals the
one-token call's (whose workgroups route for themselves, and which the oracle
tests pin) bit for bit, in the layouts where the groups can go wrong: every
token on the same experts (second groups of 1 and of 8 tokens), two experts of
a token in one slot, slots outside the pool, no shared expert, pools beyond the
first-occurrence table, every expert-count form of the top-k."""
import sys

import pytest

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _layer(gpu, H, I, E, k, *, cap=None, tied=False, shared=True, table=None, zipf=1.0):
    import torch
    from vates_amd.moe import MoELayer
    from vates_amd.workload import synth_layer
    w = synth_layer(6, 0, hidden=H, inter=I, num_experts=E, cap=cap, zipf_alpha=zipf, device=gpu)
    if tied:
        for t in (w.router.weight, w.router.scales, w.router.biases):
            t.zero_()
    return MoELayer(w.router, w.gate, w.up, w.down, top_k=k, router_bits=8,
                    shared_gate=w.sh_gate if shared else None, shared_up=w.sh_up if shared else None,
                    shared_down=w.sh_down if shared else None, shared_expert_gate=w.sgate if shared else None,
                    slot_table=torch.tensor(table, dtype=torch.int32, device=gpu) if table else w.table,
                    router_logit_bias=None if tied else w.bias, norm_weight=w.norm)


@pytest.mark.parametrize("T", [9, 13, 16])
@pytest.mark.parametrize("kw", [
    dict(H=2048, I=512, E=512, k=10), dict(H=512, I=64, E=64, k=4, tied=True),
    dict(H=1024, I=128, E=128, k=8, cap=5), dict(H=512, I=192, E=256, k=10, shared=False, zipf=2.0),
    dict(H=512, I=64, E=64, k=6, table=[i - 3 if i % 2 else i + 40 for i in range(64)]),
    dict(H=512, I=64, E=1024, k=10, cap=1100)], ids=lambda kw: "-".join(f"{a}{b}" for a, b in kw.items() if a != "table"))
def test_groups_equal_single_tokens(gpu, T, kw):
    import torch
    from vates_amd._lib import VMI_STATUS_BAD_SLOT
    from vates_amd.moe import workspace_status
    from vates_amd.synth import synth_bf16
    log(f"groups T={T} {kw}")
    kw = dict(kw)
    H, k = kw["H"], kw["k"]
    layer = _layer(gpu, **kw)
    x = synth_bf16(6, 100 + T, (T, H), device=gpu)
    ids = torch.empty((T, k), dtype=torch.int32, device=gpu)
    sc = torch.empty((T, k), dtype=torch.float32, device=gpu)
    ws = torch.zeros(layer.workspace_bytes(T), dtype=torch.uint8, device=gpu)
    out = layer(x, residual=x, ids_out=ids, scores_out=sc, ws=ws)
    i1, s1 = torch.empty_like(ids), torch.empty_like(sc)
    ws1 = torch.zeros(layer.workspace_bytes(1), dtype=torch.uint8, device=gpu)
    rows = [layer(x[t:t + 1], residual=x[t:t + 1], ids_out=i1[t:t + 1], scores_out=s1[t:t + 1], ws=ws1) for t in range(T)]
    assert torch.equal(ids, i1) and torch.equal(sc, s1)
    assert torch.equal(out.view(torch.int16), torch.cat(rows).view(torch.int16))
    flags = workspace_status(ws)
    assert flags == workspace_status(ws1)
    assert bool(flags & VMI_STATUS_BAD_SLOT) == ("table" in kw)
