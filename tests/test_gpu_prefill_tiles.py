"""Expert-major prefill at the edges of its dispatch: 64-route tiles (up to 64
routes per expert on average) and 128-route ones, the router's split of K, and
the one-workgroup and two-launch forms of the route grouping.  Bars as in
test_gpu_prefill.py.
"""
import numpy as np
import pytest

from test_gpu_prefill import _case, _check_against_oracle, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,E,k,T", [
    (512, 128, 64, 4, 17),      # a few routes a tile, four parts of K in the router (two groups each)
    (512, 64, 64, 1, 63),       # one group of down, one 64-column block
    (1024, 320, 64, 4, 128),    # odd group count in down, a partial last 128-column block
    (512, 128, 64, 4, 1024),    # 64 routes per expert: the last small-tile size ...
    (512, 128, 64, 4, 1025),    # ... and the first large-tile one
    (512, 320, 64, 4, 1100),    # large tiles with a partial last 256-column block
    (512, 64, 128, 8, 1024),    # 8192 routes: the last one-workgroup grouping ...
    (512, 64, 128, 8, 1025),    # ... and the first in two launches, a full 64-route tile count
])
def test_prefill_dispatch_edges(gpu, orc, H, I, E, k, T):
    import torch
    log(f"case: prefill H={H} I={I} E={E} k={k} T={T}")
    w, moe, x, out, ids, sc = _case(gpu, orc, T, H=H, I=I, E=E, k=k, zipf_alpha=0.5)
    counts = np.bincount(ids.cpu().numpy().ravel(), minlength=E)
    log(f"routes per expert: {counts.min()} .. {counts.max()}")
    _check_against_oracle(orc, w, x, out, ids, sc, k, True, f"H={H} I={I} T={T}")
    again = moe.prefill(x, residual=x)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16)), "not bit-deterministic"


@pytest.mark.parametrize("H,E", [(512, 128), (1024, 256), (2048, 512)])
def test_prefill_routing_does_not_depend_on_the_length(gpu, orc, H, E):
    """A token's experts and scores are the same bits in prompts on either side
    of the lengths at which the router's split of K changes."""
    import torch
    from vates_amd.synth import synth_bf16
    from vates_amd.workload import make_layer, synth_layer
    moe = make_layer(synth_layer(13, 0, hidden=H, inter=64, num_experts=E, zipf_alpha=0.5, device=gpu), top_k=4)
    x = synth_bf16(13, 77, (8300, H), device=gpu)
    first = None
    for T in (1, 60, 1000, 1025, 2049, 8300):
        log(f"case: prefill routing H={H} E={E} T={T}")
        ids = torch.empty((T, 4), dtype=torch.int32, device=gpu)
        sc = torch.empty((T, 4), dtype=torch.float32, device=gpu)
        moe.prefill(x[:T], ids_out=ids, scores_out=sc)
        if first is not None:
            n = first[0].shape[0]
            assert torch.equal(ids[:n], first[0]) and torch.equal(sc[:n], first[1])
        first = (ids, sc)
