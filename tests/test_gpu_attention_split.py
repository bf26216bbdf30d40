"""The chunk kernel's splits: 2- and 4-block chunks of short caches and the query
rows of a batch over several workgroups.  Bars as in test_gpu_attention.py: the
oracle's result, and bit equality between a batch, its tokens as single steps
and the paths of a tree (a token's result depends on the cache capacity
alone).  With 2 kv heads and 256 CUs, chunks are 2 blocks up to 3264 positions of
capacity, 4 up to 6528, 8 above.
"""
import pytest

from oracle.torch_bridge import u16
from test_gpu_attention import (assert_close, log, make_attention, test_attention_batch_equals_steps as batch_equals_steps,
                                test_attention_layer_parity as layer_parity,
                                test_attention_position_on_device as position_on_device,
                                test_attention_tree_equals_paths as tree_equals_paths)

pytestmark = pytest.mark.gpu


# first positions, a batch across a chunk boundary, both sides of each capacity; T = 3, 5 and 8 take
# 2, 3 and 4 row tiles of 16
@pytest.mark.parametrize("T,pos0,max_len", [(8, 0, 32), (3, 61, 64), (8, 60, 3264), (5, 3200, 3264), (8, 3288, 3296),
                                            (3, 126, 6528), (8, 6520, 6528), (8, 6552, 6560), (5, 255, 6560),
                                            (8, 13000, 16384), (8, 31000, 32768)])
def test_attention_split_parity(gpu, orc, T, pos0, max_len):
    layer_parity(gpu, orc, T, pos0, max_len)


@pytest.mark.parametrize("pos0,max_len", [(62, 3264), (126, 6528), (254, 6560), (12000, 16384)])
def test_attention_split_bit_equality(gpu, orc, pos0, max_len):
    batch_equals_steps(gpu, orc, pos0, max_len)
    position_on_device(gpu, pos0, max_len)
    tree_equals_paths(gpu, pos0, max_len)


@pytest.mark.parametrize("T", [5, 8])
def test_attention_split_full_batch_equals_steps(gpu, T):
    """Four row tiles, each in a workgroup of its own, against single tokens."""
    import torch
    from vates_amd.synth import synth_bf16
    for pos0, max_len in ((60, 3264), (700, 6528), (9000, 12288)):
        log(f"case: attention T={T} vs single steps pos0={pos0} max_len={max_len}")
        layer, _ = make_attention(gpu, 85)
        c1, c2 = layer.new_cache(max_len), layer.new_cache(max_len)
        for c in (c1, c2):
            c.write(0, synth_bf16(85, 20, (2, pos0, 256), device=gpu), synth_bf16(85, 21, (2, pos0, 256), device=gpu))
            c.length = pos0
        x = synth_bf16(85, 30, (T, 2048), device=gpu)
        batch = layer(x, c1)
        steps = torch.cat([layer(x[t:t + 1].contiguous(), c2) for t in range(T)])
        assert torch.equal(c1.k.view(torch.int16), c2.k.view(torch.int16))
        assert torch.equal(c1.v.view(torch.int16), c2.v.view(torch.int16))
        assert torch.equal(batch.view(torch.int16), steps.view(torch.int16))


# 48 rows (5 or 6 tokens of 8 heads) in tiles of 32 where 86 to 96 workgroups run: the second tile ends
# behind the rows of its chunk.  45, 48 (the whole capacity), 46 and 45 chunks of 2 kv heads, in chunks of 2, 4 and 8 blocks
@pytest.mark.parametrize("T", [5, 6])
@pytest.mark.parametrize("pos0,max_len", [(2810, 3072), (3066, 3072), (5800, 6528), (11500, 16384)])
def test_attention_part_row_tile_equals_steps(gpu, T, pos0, max_len):
    import torch
    from vates_amd.synth import synth_bf16
    log(f"case: attention T={T} vs single steps pos0={pos0} max_len={max_len}")
    layer, _ = make_attention(gpu, 86)
    c1, c2, c3 = (layer.new_cache(max_len) for _ in range(3))
    for c in (c1, c2, c3):
        c.write(0, synth_bf16(86, 20, (2, pos0, 256), device=gpu), synth_bf16(86, 21, (2, pos0, 256), device=gpu))
        c.length = pos0
    x = synth_bf16(86, 30, (T, 2048), device=gpu)
    batch = layer(x, c1)
    on_device = layer(x, c2, pos_device=torch.tensor([pos0], dtype=torch.int32, device=gpu))
    steps = torch.cat([layer(x[t:t + 1].contiguous(), c3) for t in range(T)])
    assert torch.equal(batch.view(torch.int16), steps.view(torch.int16))
    assert torch.equal(on_device.view(torch.int16), steps.view(torch.int16))
    for c in (c1, c2):
        assert torch.equal(c.k.view(torch.int16), c3.k.view(torch.int16))
        assert torch.equal(c.v.view(torch.int16), c3.v.view(torch.int16))


@pytest.mark.parametrize("paths,span,pos0,max_len", [(3, 5, 1000, 2048), (2, 6, 1500, 2048)])
def test_attention_part_row_tile_of_a_tree(gpu, paths, span, pos0, max_len):
    """The same tiles over a tree (3 x 16 and 2 x 24 chunks of 2 kv heads): the rows behind a path's are the next path's."""
    import torch
    from vates_amd.synth import synth_bf16
    log(f"case: attention tree {paths} x {span} vs paths pos0={pos0} max_len={max_len}")
    layer, _ = make_attention(gpu, 87)
    base = layer.new_cache(max_len)
    base.write(0, synth_bf16(87, 20, (2, pos0, 256), device=gpu), synth_bf16(87, 21, (2, pos0, 256), device=gpu))
    base.length = pos0
    x = synth_bf16(87, 30, (paths * span, 2048), device=gpu)
    tree = layer.tree(x, base, paths, pos0=pos0)
    for p in range(paths):
        c = layer.new_cache(max_len)
        c.k.copy_(base.k)
        c.v.copy_(base.v)
        rows = slice(p * span, (p + 1) * span)
        alone = torch.cat([layer(x[rows][t:t + 1].contiguous(), c, pos0=pos0 + t) for t in range(span)])
        assert torch.equal(tree[rows].view(torch.int16), alone.view(torch.int16)), p


@pytest.mark.parametrize("block,max_len", [(64, 3264), (128, 6528)])
def test_attention_keeps_sums_of_short_chunks(gpu, orc, block, max_len):
    """Keys of zeros (equal scores) and values a + b, -a, -b in chunks of their
    own: the output is the new token's value and what is left of the others'
    sums, a hundred times larger.  bf16 partial outputs of 64 or 128 keys would leave
    about a fifth of the result; the bar is the layer's (test_gpu_attention.py)."""
    import torch
    from vates_amd.synth import synth_bf16
    log(f"case: attention over cancelling chunks of {block} max_len={max_len}")
    layer, A = make_attention(gpu, 88)
    n = 3 * block
    a, b = (torch.randint(-64, 65, (2, block, 256), generator=torch.Generator(gpu).manual_seed(i), device=gpu) for i in (1, 2))
    values = torch.cat([a + b, -a, -b], 1).to(torch.bfloat16)  # whole numbers below 256: exact
    cache = layer.new_cache(max_len)
    cache.write(0, torch.zeros((2, n, 256), dtype=torch.bfloat16, device=gpu), values)
    x = (synth_bf16(88, 30, (1, 2048), device=gpu).float() * 2.0 ** -10).to(torch.bfloat16)
    k0, v0 = u16(cache.keys(0, n + 1)).copy(), u16(cache.values(0, n + 1)).copy()
    out = layer(x, cache, pos0=n)
    ref, _, _ = orc.attention_layer(u16(x), A, n, k0, v0)
    assert_close(orc.bf16_to_f32(u16(out).reshape(1, -1)), ref, "cancelling chunks")


def test_attention_workspace_covers_shorter_caches(gpu):
    """A workspace sized for a capacity holds every shorter one's call: the chunk
    count is not monotonic in the capacity, the size is."""
    import vates_amd._lib as L
    lib = L.load()
    size = [lib.vmi_attention_layer_workspace_bytes(8, 2048, 16, 2, 32 * b) for b in range(1, 1300)]
    assert all(a <= b for a, b in zip(size, size[1:]))
