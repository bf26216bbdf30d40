"""The prompt kernels against the CPU oracle (float64), and whole prompts at
the lengths where other kernels take over: pieces of the delta rule, 128-row
attention tiles, more than one block, two callers at once.  Bars of the layers
as in test_gpu_attention.py, test_gpu_gdn.py and test_gpu_prefill.py (relative
L2 1e-2, cosine 0.9999, max 1e-2 of the row's largest, per token)."""
import threading

import numpy as np
import pytest

from test_gpu_attention import make_attention
from test_gpu_gdn import make_gdn
from test_gpu_prefill import _case, assert_close, log
from test_gpu_prompt import _caches_close, rel

from oracle.torch_bridge import layer_np, u16

pytestmark = pytest.mark.gpu


# a whole prompt across tiles and cache blocks, and one that continues off every edge
@pytest.mark.parametrize("T,pos0,H", [(150, 0, 512), (70, 37, 2048)])
def test_attention_prompt_parity(gpu, orc, T, pos0, H):
    from vates_amd.synth import synth_bf16
    log(f"case: attention prompt H={H} T={T} pos0={pos0}")
    layer, A = make_attention(gpu, 81, H=H)
    cache = layer.new_cache(pos0 + T)
    if pos0:
        cache.write(0, synth_bf16(81, 20, (2, pos0, 256), device=gpu), synth_bf16(81, 21, (2, pos0, 256), device=gpu))
    x = synth_bf16(81, 22, (T, H), device=gpu)
    k0, v0 = u16(cache.keys(0, pos0 + T)).copy(), u16(cache.values(0, pos0 + T)).copy()
    out = layer.prompt(x, cache, pos0=pos0)
    ref, kn, vn = orc.attention_layer(u16(x), A, pos0, k0, v0)
    assert_close(orc.bf16_to_f32(u16(out).reshape(T, -1)), ref, f"attention prompt T={T}")
    for got, want in ((cache.keys(pos0, pos0 + T), kn), (cache.values(pos0, pos0 + T), vn)):
        got = orc.bf16_to_f32(u16(got).reshape(2, T, 256)).transpose(1, 0, 2)
        assert np.all(np.abs(got - want).max(axis=2) <= 2 ** -7 * np.abs(want).max(axis=2))


@pytest.mark.parametrize("T,prefix", [(60, 0), (45, 19), (361, 5)])  # the last: 352 tokens in pieces
def test_gdn_prompt_parity(gpu, orc, T, prefix):
    from vates_amd.synth import synth_bf16
    log(f"case: gdn prompt T={T} after {prefix} positions")
    layer, G = make_gdn(gpu, 91, H=512, n_k=4, n_v=8)
    cache = layer.new_cache(8)
    if prefix:
        layer.prompt(synth_bf16(91, 100, (prefix, 512), device=gpu), cache, pos0=0)
    conv = orc.bf16_to_f32(u16(cache.conv_rows(prefix))).astype(np.float64)
    state = cache.state_before(prefix).double().cpu().numpy()
    x = synth_bf16(91, 7, (T, 512), device=gpu)
    out = layer.prompt(x, cache, pos0=prefix)
    ref, _, states = orc.gdn_layer(u16(x), G, conv_in=conv, state_in=state if prefix else None)
    assert_close(orc.bf16_to_f32(u16(out).reshape(T, -1)), ref, f"gdn prompt T={T}")
    for p in range(T - 8, T + 1):
        got, want = cache.state_before(prefix + p).double().cpu().numpy(), states[p - 1]
        assert np.linalg.norm(got - want) <= 1e-2 * np.linalg.norm(want), p


@pytest.mark.parametrize("H,I,E,k,T", [(512, 128, 64, 4, 70), (1024, 320, 64, 4, 150), (2048, 512, 512, 10, 96)])
def test_moe_prompt_parity(gpu, orc, H, I, E, k, T):
    """The experts, scores and weights against the oracle on the prefill's own
    routing (the same bits, test_gpu_prompt.py), which test_gpu_prefill.py pins."""
    log(f"case: moe prompt H={H} I={I} E={E} k={k} T={T}")
    w, moe, x, _, ids, sc = _case(gpu, orc, T, H=H, I=I, E=E, k=k)
    out = moe.prompt(x, residual=x)
    ref, _ = orc.moe_layer_routed(u16(x), layer_np(w, k, True), ids.cpu().numpy(), sc.cpu().numpy(), residual=True)
    assert_close(orc.bf16_to_f32(u16(out).reshape(T, -1)), ref, f"moe prompt T={T}")


def _model(gpu, n_heads=4):
    from vates_amd.workload import synth_spec_model
    return synth_spec_model(5, n_layers=2, attn_every=2, hidden=512, inter=128, num_experts=64, top_k=4, vocab=2000,
                            n_heads=n_heads, n_k_heads=4, n_v_heads=8, device=gpu)


def _prompt(gpu, P):
    import torch
    return torch.randint(0, 2000, (P,), dtype=torch.int32, device=gpu, generator=torch.Generator(gpu).manual_seed(P))


# the delta rule in pieces; two blocks of 2100, each with 128-row attention tiles
@pytest.mark.parametrize("P,n_heads", [(420, 4), (4200, 16)])
def test_long_prefill_equals_verify_batches(gpu, P, n_heads, monkeypatch):
    from vates_amd import decode
    from vates_amd.mtp import MTPDrafter
    log(f"case: prompt of {P} tokens through the model")
    model, prompt = _model(gpu, n_heads), _prompt(gpu, P)
    runs = []
    for least in (10 ** 9, 16):
        monkeypatch.setattr(decode, "PROMPT_MIN", least)
        caches, drafter = model.new_caches(P + 9), MTPDrafter(model.mtp, P + 9)
        runs.append((caches, drafter, decode.prefill(model, prompt, caches, drafter)[1]))
    (A, da, ha), (B, db, hb) = runs
    _caches_close(model, A, B, P)
    assert da.cache.length == db.cache.length == P - 1
    assert rel(db.cache.keys(), da.cache.keys()) <= 0.03 and rel(db.cache.values(), da.cache.values()) <= 0.03
    assert rel(hb, ha) <= 0.03


def test_prompts_of_two_threads(gpu):
    """Two prompts through one model at once, a thread and a stream each, give
    what they give one after the other, bit for bit."""
    import torch
    from vates_amd import decode
    from vates_amd.mtp import MTPDrafter
    log("case: two prompts at once")
    model = _model(gpu)
    model.layers[0].moe.prefill_tables()
    prompts = [_prompt(gpu, P) for P in (700, 431)]

    def state():
        return model.new_caches(800), MTPDrafter(model.mtp, 800)

    def run(prompt, caches, drafter):
        am, h = decode.prefill(model, prompt, caches, drafter)
        return [am, h, caches[0].state, caches[0].conv, caches[1].k, caches[1].v, drafter.cache.k, drafter.cache.v]

    want = [run(p, *state()) for p in prompts]
    states = [[state() for _ in prompts] for _ in range(3)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in prompts]
    for turn in states:
        got, start = [None, None], threading.Barrier(2)

        def work(i):
            with torch.cuda.stream(streams[i]):
                start.wait()
                got[i] = run(prompts[i], *turn[i])
                streams[i].synchronize()

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for g, w in zip(got, want):
            assert g is not None
            for a, b in zip(g, w):
                assert torch.equal(a, b)
    assert model.layers[0].moe.desc.prefill_tables
