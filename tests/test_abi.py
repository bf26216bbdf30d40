"""The C ABI library loads on the CPU and exports every symbol include/vmi.h
declares; argument validation runs without touching a device."""
import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared_functions():
    text = (ROOT / "include" / "vmi.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vmi_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    import vates_amd._lib as L
    if not L.LIB_PATH.exists():
        pytest.fail("libvmi.so is not built (run __graft_entry__.build())")
    return L.load()


def test_every_declared_symbol_is_exported(lib):
    names = declared_functions()
    assert len(names) >= 10
    for n in names:
        assert hasattr(lib, n), n


def test_python_binding_covers_header():
    import vates_amd._lib as L
    assert sorted(L.exported_names()) == declared_functions()


def test_version_and_workspace_queries(lib):
    assert lib.vmi_version() == 1
    # at least the per-(distinct slot, token) bf16 activation operands of the down projection,
    # and the fp32 path's activation and output rows per pair
    assert lib.vmi_fused_moe_slots_workspace_bytes(4, 10, 2048, 512) >= (4 * 10 + 1) * 4 * 512 * 2
    assert lib.vmi_fused_moe_slots_workspace_bytes(4, 10, 2048, 512) >= 4 * 10 * (512 + 2048) * 4
    # the whole layer also holds the router logits [T, E]
    assert lib.vmi_moe_layer_workspace_bytes(4, 10, 2048, 512, 512) >= (4 * 10 + 1) * 4 * 512 * 2 + 4 * 512 * 4
    assert lib.vmi_fused_moe_slots_workspace_bytes(0, 10, 2048, 512) == 0


def test_prompt_forms_are_the_documented_ones(lib):
    """The prompt queries answer 0 for exactly the head counts include/vmi.h
    leaves out (k_pr_wy's grid takes four value heads a workgroup)."""
    from vates_amd._lib import MoeLayerDesc, QMat
    from vates_amd.attention import AttnDesc
    from vates_amd.gdn import GdnDesc
    q = QMat(4096, 4096, 4096)
    for n in range(1, 80):
        a = AttnDesc()
        a.hidden, a.n_heads, a.n_kv_heads, a.head_dim, a.rope_dim, a.bits, a.group = 512, n, 1, 256, 64, 4, 64
        a.q_proj = a.k_proj = a.v_proj = a.o_proj = q
        a.input_norm = a.q_norm = a.k_norm = 4096
        assert bool(lib.vmi_attention_prompt_workspace_bytes(ctypes.byref(a), 40)) == (n % 2 == 0 and n <= 16), n
        g = GdnDesc()
        g.hidden, g.n_k_heads, g.n_v_heads, g.head_k_dim, g.head_v_dim, g.bits, g.group = 512, 1, n, 128, 128, 4, 64
        g.in_proj_qkvz = g.in_proj_ba = g.out_proj = q
        g.input_norm = g.conv_weight = g.A_log = g.dt_bias = g.norm_weight = 4096
        assert bool(lib.vmi_gdn_prompt_workspace_bytes(ctypes.byref(g), 40)) == (n % 4 == 0 and n <= 32), n
        m = MoeLayerDesc()
        m.hidden, m.inter, m.num_experts, m.top_k, m.group, m.bits, m.router_bits, m.cap = 512, 64, n, 4, 64, 4, 8, 64
        m.router = m.gate = m.up = m.down = q
        assert bool(lib.vmi_moe_prompt_workspace_bytes(ctypes.byref(m), 40)) == (n == 64), n
    m.num_experts, m.cap = 64, 1025
    assert lib.vmi_moe_prompt_workspace_bytes(ctypes.byref(m), 40) == 0
    m.cap, m.down = 64, QMat(4096, 4100, 4096)
    assert lib.vmi_moe_prompt_workspace_bytes(ctypes.byref(m), 40) == 0


@pytest.mark.parametrize("k,hidden,inter,experts,cap", [
    (10, 2048, 512, 512, 512), (1, 512, 64, 1024, 1024), (16, 1024, 320, 64, 9), (4, 512, 128, 64, 64), (8, 2048, 64, 1024, 5)])
def test_prefill_workspace_grows_with_the_prompt(lib, k, hidden, inter, experts, cap):
    """A workspace of a longer prompt takes every shorter one, across the lengths
    at which the router's parts and the expert tiles change."""
    size = [lib.vmi_moe_prefill_workspace_bytes(T, k, hidden, inter, experts, cap, 8) for T in range(1, 9000)]
    assert all(a <= b for a, b in zip(size, size[1:]))


def test_invalid_arguments_rejected_before_any_device_call(lib):
    import vates_amd._lib as L
    q = L.QMat(None, None, None)
    rc = lib.vmi_fused_moe_slots(None, 0, None, None, q, q, q, 0, 10, 2048, 512, 64, 4, 512, None, 0, None, 0, None)
    assert rc == L.VMI_ERR_INVALID
    assert b"T=0" in lib.vmi_last_error()
    rc = lib.vmi_fused_moe_slots(None, 0, None, None, q, q, q, 4, 10, 2048, 512, 32, 4, 512, None, 0, None, 0, None)
    assert rc == L.VMI_ERR_UNSUPPORTED
    rc = lib.vmi_fused_moe_slots(None, 0, None, None, q, q, q, 17, 1, 2048, 512, 64, 4, 512, None, 0, None, 0, None)
    assert rc == L.VMI_ERR_UNSUPPORTED
    rc = lib.vmi_moe_layer(None, None, 4, None, None, None, None, None, 0, None)
    assert rc == L.VMI_ERR_INVALID
    # the prefill tables: two fp16 halves per (row, group) of gate, up and down
    # for every slot and the shared expert, plus a factor per row
    assert lib.vmi_moe_prefill_tables_bytes(2048, 512, 512) >= 513 * (2 * 512 * 32 + 2048 * 8) * 4
    assert lib.vmi_moe_prefill_tables_bytes(2048, 100, 512) == 0
    assert lib.vmi_moe_prefill_tables(None, None, 0, None) == L.VMI_ERR_INVALID
    d = L.MoeLayerDesc()
    d.hidden, d.inter, d.cap, d.bits, d.group = 2048, 512, 512, 4, 64
    rc = lib.vmi_moe_prefill_tables(ctypes.byref(d), None, 0, None)
    assert rc == L.VMI_ERR_INVALID and b"scales" in lib.vmi_last_error()
    rc = lib.vmi_spec_commit(None, None, 4, 1, 2048, 0, None, None, None, None, None, None, None)
    assert rc == L.VMI_ERR_INVALID and b"K=0" in lib.vmi_last_error()
    rc = lib.vmi_spec_commit(None, None, 0, 1, 2048, 3, None, None, None, None, None, None, None)
    assert rc == L.VMI_ERR_INVALID and b"rows=0" in lib.vmi_last_error()
    rc = lib.vmi_spec_commit(None, None, 4, 1, 2048, 3, None, None, None, None, None, None, None)
    assert rc == L.VMI_ERR_INVALID


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    import vates_amd._lib as L
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L, "LIB_PATH", tmp_path / "libvmi.so")
    with pytest.raises(L.VmiError):
        L.load()
