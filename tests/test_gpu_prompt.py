"""GPU tests of the prompt kernels (vmi_attention_prompt, vmi_gdn_prompt,
vmi_qgemm, decode.prefill's blocks) against the verify kernels run over the
same tokens in batches of at most eight, which the oracle tests pin
(tests/test_gpu_attention.py, tests/test_gpu_gdn.py): the two differ by the
order of fp32 sums, so bf16 results differ by at most one rounding step
(2^-8 of the value) here and there: relative L2 well below 2^-8 = 3.9e-3.

Sizes: one token past a verify batch, the edges of the 32-position cache
block, of the 16-token scan piece, of the 64- and 128-token GEMM tiles and of the
128-row attention tile, a block continuing at a position off every edge, head
counts other than the default, rotary widths of every form."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BF16_REL = 2.0 ** -8


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


def branch_close(got, want, x):
    """out = bf16(x + branch): the branches agree within 2^-8 of their norm
    (their bf16 inputs round alike but for ties moved by fp32 order), and the
    sum's own rounding adds at most one step, 2^-8 of the value, where the
    branches straddle a rounding boundary."""
    got, want, x = got.double(), want.double(), x.double()
    assert float((got - want).norm()) <= BF16_REL * float((want - x).norm()) + 0.5 * BF16_REL * float(want.norm())
    assert float(((got - want).abs() - BF16_REL * want.abs()).max()) <= 0.05 * float((want - x).abs().max())


def _attention(gpu, n_heads, n_kv, hidden, rope):
    from vates_amd.attention import AttentionLayer
    from vates_amd.synth import synth_proj
    from vates_amd.workload import bf16_norm
    p = lambda i, n, k: synth_proj(9, 8 + i, 1, n, k, device=gpu)  # noqa: E731
    return AttentionLayer(p(0, n_heads * 512, hidden), p(1, n_kv * 256, hidden), p(2, n_kv * 256, hidden),
                          p(3, hidden, n_heads * 256), bf16_norm(9, 1, hidden, gpu), bf16_norm(9, 2, 256, gpu),
                          bf16_norm(9, 3, 256, gpu), n_heads=n_heads, n_kv_heads=n_kv, rope_dim=rope)


@pytest.mark.parametrize("n_heads,n_kv,hidden,rope,T,start", [
    (16, 2, 2048, 64, 9, 0), (16, 2, 2048, 64, 17, 0), (16, 2, 2048, 64, 33, 37), (16, 2, 2048, 64, 129, 0),
    (16, 2, 2048, 64, 300, 61), (8, 4, 1024, 128, 70, 5), (4, 2, 512, 256, 64, 32), (2, 2, 512, 40, 131, 1),
    (6, 1, 512, 0, 45, 3),
    (16, 2, 512, 64, 2033, 0)])  # the fewest tokens whose 128-row attention tiles give 256 CUs one each
def test_attention_prompt_equals_verify_batches(gpu, n_heads, n_kv, hidden, rope, T, start):
    import torch
    from vates_amd.synth import synth_bf16
    log(f"attention prompt heads {n_heads}/{n_kv} hidden {hidden} rope {rope} T {T} start {start}")
    layer = _attention(gpu, n_heads, n_kv, hidden, rope)
    x = synth_bf16(9, 77, (start + T, hidden), device=gpu)
    a, b = layer.new_cache(start + T + 7), layer.new_cache(start + T + 7)
    for c in (a, b):  # stale contents past the block are never read
        c.k.fill_(float("nan"))
        c.v.fill_(float("nan"))
    outs = []
    for s in range(0, start + T, 8):
        outs.append(layer(x[s:s + 8], a, pos0=s))
    want = torch.cat(outs)
    if start:
        layer.prompt(x[:start], b, pos0=0)
    got = layer.prompt(x[start:], b, pos0=start)
    assert b.length == start + T
    branch_close(got, want[start:], x[start:])
    for name in ("keys", "values"):
        assert rel(getattr(b, name)(), getattr(a, name)()) <= BF16_REL
    kv = layer.new_cache(start + T + 7)
    assert layer.prompt(x, kv, pos0=0, keys_only=True) is None
    assert rel(kv.keys(), a.keys()) <= BF16_REL and rel(kv.values(), a.values()) <= BF16_REL


@pytest.mark.parametrize("n_heads,n_kv,T,start", [(16, 2, 200, 0), (16, 2, 131, 37), (2, 2, 140, 3), (16, 2, 2040, 0)])
def test_attention_prompt_keeps_tokens_before_a_nan(gpu, n_heads, n_kv, T, start):
    """A token that is not finite leaves every token before it as it was, bit
    for bit, in its tile of query rows and its cache block too (2040 tokens: 128-row tiles)."""
    import torch
    from vates_amd.synth import synth_bf16
    log(f"attention prompt with a NaN token, heads {n_heads}/{n_kv} T {T} start {start}")
    layer = _attention(gpu, n_heads, n_kv, 512, 64)
    x = synth_bf16(9, 79, (start + T, 512), device=gpu)

    def go(x):
        cache = layer.new_cache(start + T)
        if start:
            layer.prompt(x[:start], cache, pos0=0)
        return layer.prompt(x[start:], cache, pos0=start)

    want = go(x)
    for bad in (0, 13, 32, T - 9, T - 1):
        y = x.clone()
        y[start + bad] = float("nan")
        got = go(y)
        assert torch.equal(got[:bad].view(torch.int16), want[:bad].view(torch.int16)), bad
        assert bool(torch.isnan(got[bad:].float()).any(1).all()), bad


@pytest.mark.parametrize("n_k,n_v,hidden,T,start,slots", [
    (16, 32, 2048, 9, 0, 9), (16, 32, 2048, 17, 0, 9), (16, 32, 2048, 33, 5, 9), (16, 32, 2048, 130, 2, 6),
    (4, 4, 512, 64, 31, 9), (2, 8, 1024, 31, 1, 3), (4, 8, 512, 48, 64, 20),
    (4, 8, 512, 264, 0, 9), (4, 8, 512, 265, 0, 9), (2, 4, 512, 288, 3, 9), (16, 32, 2048, 301, 0, 9),
    # pieces of 16 tokens: one token short of the fewest (336 of 345), the fewest, counts off the rotation of three, a wide ring
    (4, 8, 512, 344, 0, 9), (4, 8, 512, 345, 0, 9), (2, 4, 512, 365, 3, 9), (16, 32, 2048, 380, 0, 9), (4, 4, 512, 530, 40, 170),
    (4, 4, 512, 450, 40, 170)])
def test_gdn_prompt_equals_verify_batches(gpu, n_k, n_v, hidden, T, start, slots):
    import torch
    from vates_amd.gdn import GdnCache
    from vates_amd.synth import synth_bf16
    from vates_amd.workload import synth_gdn
    log(f"gdn prompt heads {n_k}/{n_v} hidden {hidden} T {T} start {start} slots {slots}")
    layer = synth_gdn(3, 1, hidden=hidden, n_k_heads=n_k, n_v_heads=n_v, device=gpu)
    x = synth_bf16(3, 78, (start + T, hidden), device=gpu)
    a, b = (GdnCache(n_k, n_v, slots, gpu) for _ in range(2))
    outs = []
    step = min(8, slots - 1)
    for s in range(0, start + T, step):
        outs.append(layer(x[s:s + step], a, pos0=s))
    want = torch.cat(outs)
    if start:
        layer.prompt(x[:start], b, pos0=0)
    got = layer.prompt(x[start:], b, pos0=start)
    end = start + T
    assert b.length == end
    branch_close(got, want[start:], x[start:])
    assert rel(b.conv_rows(end), a.conv_rows(end)) <= BF16_REL
    n = min(end, 32)
    assert rel(torch.stack([b.conv[p % 32] for p in range(end - n, end)]),
               torch.stack([a.conv[p % 32] for p in range(end - n, end)])) <= BF16_REL
    # the states before the last n_slots positions, as a trim after the prompt may need them
    for p in range(max(1, end - slots + 1), end + 1):
        assert rel(b.state_before(p), a.state_before(p)) <= BF16_REL, p


def test_gdn_prompt_keeps_tokens_before_a_nan(gpu):
    """A token that is not finite leaves every token before it as it was, those of its own piece of 16 too."""
    import torch
    from vates_amd.gdn import GdnCache
    from vates_amd.synth import synth_bf16
    from vates_amd.workload import synth_gdn
    log("gdn prompt with a NaN token")
    layer = synth_gdn(3, 1, hidden=512, n_k_heads=4, n_v_heads=8, device=gpu)
    x = synth_bf16(3, 79, (400, 512), device=gpu)
    want = layer.prompt(x, GdnCache(4, 8, 9, gpu), pos0=0)
    for bad in (5, 70, 299, 399):
        y = x.clone()
        y[bad] = float("nan")
        got = layer.prompt(y, GdnCache(4, 8, 9, gpu), pos0=0)
        branch_close(got[:bad], want[:bad], x[:bad])
        assert bool(torch.isnan(got[bad:].float()).any(1).all())


# the 32 x 32, 64 x 64, 64 x 128 and 128 x 256 tiles of the GEMM, each with part tiles
# of both dimensions, one to eight blocks of four stages, and several rounds of workgroups
@pytest.mark.parametrize("T,K,N", [(17, 512, 16), (64, 1024, 129), (65, 2048, 2048), (128, 4096, 2048),
                                   (129, 1536, 333), (1000, 512, 4096), (33, 512, 8193), (97, 3584, 5000),
                                   (321, 2560, 2049), (515, 512, 9217), (1025, 3072, 2305)])
def test_qgemm_equals_qgemv(gpu, T, K, N):
    import torch
    from vates_amd.attention import qgemm, qgemv
    from vates_amd.synth import synth_bf16, synth_proj
    log(f"qgemm T {T} K {K} N {N}")
    w = synth_proj(4, 1, 1, N, K, device=gpu)
    x = synth_bf16(4, 2, (T, K), device=gpu)
    want = torch.cat([qgemv(x[s:s + 4].contiguous(), w) for s in range(0, T, 4)])
    got = qgemm(x, w, torch.empty((T, N), dtype=torch.bfloat16, device=gpu))
    # one rounding to bf16 apart: half an ulp, 2^-9 of the value, plus fp32 sums
    assert float(((got.float() - want).abs() - 2.0 ** -8 * want.abs()).max()) <= 1e-5 * float(want.abs().max())


# a tile of one, of some and of all four 16-route blocks; intermediate sizes of one and of an odd count of groups, a
# partial last column block, and of two and four eights of groups; no shared expert; one slot for two experts; every width
@pytest.mark.parametrize("H,I,E,k,T,kw", [
    (512, 64, 64, 1, 17, {}), (1024, 320, 64, 4, 128, {}), (512, 192, 64, 4, 700, dict(cap=5)), (2048, 512, 512, 10, 200, {}),
    (512, 1024, 64, 2, 90, {}), (512, 2048, 64, 2, 300, {}), (1024, 576, 128, 6, 61, dict(shared=False))])
def test_moe_prompt_equals_prefill(gpu, H, I, E, k, T, kw):
    """vmi_moe_prompt routes as vmi_moe_prefill, bit for bit, and its exact
    weights differ from that one's fp16 ones by 2^-12 of a weight, so a row by
    the bf16 rounding of activations and partial rows: 2^-8."""
    import torch
    from vates_amd.moe import MoELayer
    from vates_amd.synth import synth_bf16
    from vates_amd.workload import synth_layer
    log(f"moe prompt H {H} I {I} E {E} k {k} T {T} {kw}")
    w = synth_layer(6, 0, hidden=H, inter=I, num_experts=E, cap=kw.get("cap"), zipf_alpha=0.5, device=gpu)
    sh = kw.get("shared", True)
    layer = MoELayer(w.router, w.gate, w.up, w.down, top_k=k, router_bits=8, shared_gate=w.sh_gate if sh else None,
                     shared_up=w.sh_up if sh else None, shared_down=w.sh_down if sh else None,
                     shared_expert_gate=w.sgate if sh else None, slot_table=w.table, router_logit_bias=w.bias, norm_weight=w.norm)
    x = synth_bf16(6, 100, (T, H), device=gpu)
    got, want = layer.prompt(x), layer.prefill(x)
    err = (got.double() - want.double()).norm(dim=1) / want.double().norm(dim=1)
    assert float(err.max()) <= BF16_REL
    assert torch.equal(layer.prompt(x).view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize("H,I,T", [(512, 64, 40), (2048, 512, 90)])
def test_moe_prompt_keeps_the_weights_bits(gpu, H, I, T):
    """Gate and up weights 8 + q 2^-9 on columns that cancel in pairs: the
    result hangs on q alone, which weights rounded to fp16 (steps of 2^-7 at 8)
    have lost.  Against the one-token kernel, whose operands are exact; the
    two round activations and partial rows to bf16 apart.  Rows whose routing has a
    near-tie may differ: at most one in twenty."""
    import torch
    from vates_amd.synth import synth_bf16
    from vates_amd.workload import make_layer, synth_layer
    log(f"moe prompt exact weights H {H} I {I} T {T}")
    w = synth_layer(7, 0, hidden=H, inter=I, num_experts=64, zipf_alpha=0.5, with_norm=False, device=gpu)
    for p in (w.gate, w.up, w.sh_gate, w.sh_up):
        p.scales.view(torch.bfloat16).fill_(2.0 ** -9)
        p.biases.view(torch.bfloat16).fill_(8.0)
    layer = make_layer(w, top_k=4)
    x = synth_bf16(7, 100, (T, H), std=4.0, device=gpu)
    x[:, 1::2] = -x[:, ::2]
    want = torch.cat([layer(x[t:t + 1].contiguous()) for t in range(T)]).double()
    err = lambda y: (y.double() - want).norm(dim=1) / want.norm(dim=1)  # noqa: E731
    got, rounded = err(layer.prompt(x)), err(layer.prefill(x))
    log(f"exact {float(got.median()):.2e}, fp16 weights {float(rounded.median()):.2e}")
    assert float(got.quantile(0.95)) <= 2 * BF16_REL
    assert float(rounded.median()) > 4 * BF16_REL


def _caches_close(model, A, B, end):
    from vates_amd.attention import KVCache
    for a, b in zip(A, B):
        if isinstance(a, KVCache):
            assert rel(b.keys(), a.keys()) <= 0.03 and rel(b.values(), a.values()) <= 0.03
        elif a is not None:
            assert rel(b.state_before(end), a.state_before(end)) <= 0.03
        if a is not None:
            assert a.length == b.length == end


@pytest.mark.parametrize("P", [17, 40, 203])
def test_prefill_blocks_equal_verify_batches(gpu, P, monkeypatch):
    """The whole call, in one block and in blocks of 64, against batches of
    eight: bf16 rounding through two layers and the routing near-ties it
    decides (a token changes one of its ten experts) stay within 3e-2."""
    import torch
    from vates_amd import decode
    from vates_amd.mtp import MTPDrafter
    from vates_amd.workload import synth_spec_model
    model = synth_spec_model(5, n_layers=2, attn_every=2, hidden=512, inter=128, num_experts=64, top_k=4, vocab=2000,
                             n_heads=4, n_k_heads=4, n_v_heads=8, device=gpu)
    prompt = torch.randint(0, 2000, (P,), dtype=torch.int32, device=gpu, generator=torch.Generator(gpu).manual_seed(P))

    def go(block, least):
        monkeypatch.setattr(decode, "PROMPT_BLOCK", block)
        monkeypatch.setattr(decode, "PROMPT_MIN", least)
        caches, drafter = model.new_caches(P + 9), MTPDrafter(model.mtp, P + 9)
        assert bool(decode._prompt_blocks(model, prompt, caches, drafter, 8)) == (least < P)
        x, h = decode.prefill(model, prompt, caches, drafter)
        return caches, drafter, x, h

    A, da, xa, ha = go(4096, 10 ** 9)
    for block in (4096, 64):
        B, db, xb, hb = go(block, 16)
        _caches_close(model, A, B, P)
        assert da.cache.length == db.cache.length == P - 1
        assert rel(db.cache.keys(), da.cache.keys()) <= 0.03 and rel(db.cache.values(), da.cache.values()) <= 0.03
        assert rel(hb, ha) <= 0.03 and xb.shape == xa.shape


def test_prefill_refuses_what_verify_batches_refuse(gpu):
    import torch
    from vates_amd import decode
    from vates_amd._lib import VmiError
    from vates_amd.workload import synth_spec_model
    model = synth_spec_model(5, n_layers=2, attn_every=2, hidden=512, inter=128, num_experts=64, top_k=4, vocab=2000,
                             n_heads=4, n_k_heads=4, n_v_heads=8, device=gpu)
    prompt = torch.zeros(40, dtype=torch.int32, device=gpu)
    with pytest.raises(VmiError):
        decode.prefill(model, prompt, model.new_caches(32))            # a KV cache too small
    with pytest.raises(VmiError):
        decode.prefill(model, prompt, model.new_caches(64), chunk=9)   # wider than the layers take
    with pytest.raises(VmiError):
        decode.prefill(model, prompt, model.new_caches(64, max_batch=4))  # a state ring too small for chunks of 8
    x, h = decode.prefill(model, prompt, model.new_caches(64, max_batch=4), chunk=4)
    assert h.shape == (1, 512)


def test_prefill_reports_where_verify_batches_do(gpu, monkeypatch):
    """A prompt's MoE status bits are read from the stream's MoE workspace, as after verify batches."""
    import torch
    from vates_amd import decode
    from vates_amd._lib import VMI_STATUS_BAD_SLOT
    from vates_amd.moe import workspace, workspace_status
    from vates_amd.workload import synth_spec_model
    model = synth_spec_model(5, n_layers=1, attn_every=1, hidden=512, inter=128, num_experts=64, top_k=4, vocab=2000,
                             n_heads=4, n_k_heads=4, n_v_heads=8, device=gpu)
    moe = model.layers[0].moe
    table = torch.full((64,), 10 ** 6, dtype=torch.int32, device=gpu)
    prompt = torch.zeros(40, dtype=torch.int32, device=gpu)
    sh = torch.cuda.current_stream().cuda_stream
    good = moe.desc.slot_table
    for least in (10 ** 9, 16):
        monkeypatch.setattr(decode, "PROMPT_MIN", least)
        ws = workspace(moe.workspace_bytes(8), gpu, sh)
        workspace_status(ws)
        decode.prefill(model, prompt, model.new_caches(64))
        assert workspace_status(ws) == 0
        moe.desc.slot_table = table.data_ptr()
        decode.prefill(model, prompt, model.new_caches(64))
        moe.desc.slot_table = good
        assert workspace_status(ws) & VMI_STATUS_BAD_SLOT
        assert workspace_status(ws) == 0


def test_prefill_gives_its_workspace_back(gpu):
    """A prompt leaves no workspace of its length behind."""
    import torch
    from vates_amd import decode, moe
    from vates_amd.workload import synth_spec_model
    model = synth_spec_model(5, n_layers=2, attn_every=2, hidden=512, inter=128, num_experts=64, top_k=4, vocab=2000,
                             n_heads=4, n_k_heads=4, n_v_heads=8, device=gpu)
    prompt = torch.zeros(3000, dtype=torch.int32, device=gpu)
    caches = model.new_caches(3000)
    decode.prefill(model, prompt[:8], caches)  # the head's and verify batches' workspaces
    kept, held = sum(t.numel() for t in moe._WORKSPACES.values()), torch.cuda.memory_allocated()
    _, last = decode.prefill(model, prompt, caches)
    del last
    assert sum(t.numel() for t in moe._WORKSPACES.values()) == kept
    assert torch.cuda.memory_allocated() <= held + (1 << 20)
