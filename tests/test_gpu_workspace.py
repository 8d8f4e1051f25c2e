"""Workspaces between the least a call accepts and what it asks for: the same results, nothing
written past the end.  The least is what the call names when it is given none."""
import ctypes
import re

import pytest
import torch

from amla import ops, synth
from amla._lib import check, lib
from amla.config import DeepSeekConfig
from amla.torch_ops import fill_mla_args
from oracle import ref_ffn as F
from oracle import ref_ops as R
from _tol import assert_parity

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CFG = DeepSeekConfig()


def _least(call):
    """call(pointer, bytes) -> status."""
    assert call(None, 0) == -2
    m = re.search(rb"needs (\d+) bytes|< (\d+) needed", lib().amla_last_error())
    return int(m.group(1) or m.group(2))


def _run(call, nbytes):
    buf = torch.full((nbytes + 4096,), 0x5A, dtype=torch.uint8, device=DEV)
    check(call(buf.data_ptr(), nbytes), "call")
    torch.cuda.synchronize()
    assert (buf[nbytes:] == 0x5A).all(), "written past the workspace"


@pytest.mark.parametrize("m,n,k", [(65, 256, 1024), (100, 1408, 2048), (300, 512, 1152)])
def test_swiglu_without_room_for_k_parts(m, n, k):
    print(f"[case] swiglu workspace m={m} n={n} k={k}", flush=True)
    w = []
    for i, (a, b) in enumerate(((n, k), (n, k), (k, n))):
        q, s = synth.quantize_fp8_blocks(synth.randn((a, b), synth.seed_of("ws", i, n, k), 0.05))
        w += [q.to(DEV), s.to(DEV)]
    x = synth.randn((m, k), synth.seed_of("ws-x", m, k), 1.0).to(torch.bfloat16).to(DEV)
    y = torch.empty(m, k, dtype=torch.bfloat16, device=DEV)
    g, gs, u, us, d, ds = [t.data_ptr() for t in w]
    call = lambda p, b: lib().amla_swiglu(x.data_ptr(), m, k, g, gs, u, us, n, d, ds, y.data_ptr(), p, b,
                                          ops._stream_ptr(x))
    want = F.swiglu(x.cpu(), *[t.cpu() for t in w])
    full, least = lib().amla_swiglu_workspace_bytes(m, k, n), _least(call)
    assert least < full, "no K parts at this size"
    for b in (full, least, (full + least) // 2):
        y.zero_()
        _run(call, b)
        assert_parity(y, want, f"swiglu m={m} in {b} bytes")
    assert call(x.data_ptr(), least - 1) == -2


@pytest.mark.parametrize("m", [65, 300])
def test_route_with_fewer_k_splits(m):
    print(f"[case] route workspace m={m}", flush=True)
    E, k, top_k = CFG.n_routed_experts, 1024, CFG.num_experts_per_tok
    x = synth.randn((m, k), synth.seed_of("wsr", m), 1.0).to(torch.bfloat16).to(DEV)
    gw = synth.randn((E, k), synth.seed_of("wsg", E), 0.05).to(torch.bfloat16).to(DEV)
    idx = torch.empty(m, top_k, dtype=torch.int64, device=DEV)
    w = torch.empty(m, top_k, device=DEV)
    call = lambda p, b: lib().amla_moe_route(x.data_ptr(), m, k, gw.data_ptr(), E, CFG.n_group, CFG.topk_group, top_k, 1,
                                             idx.data_ptr(), w.data_ptr(), p, b, ops._stream_ptr(x))
    full, least = lib().amla_moe_route_workspace_bytes(m, E), _least(call)
    assert least == m * E * 4 < full
    _run(call, full)
    i0, w0 = idx.clone(), w.clone()
    for b in (least, 2 * least + 256):
        _run(call, b)
        # fp32 sums of 1024 products in another order
        assert torch.allclose(w, w0, rtol=1e-5, atol=1e-6) and (idx == i0).float().mean() > 0.999


def test_experts_without_room_for_k_parts():
    """Few experts, 40 tokens: the skinny GEMM with its K-part sums, or the tiles without."""
    print("[case] experts workspace", flush=True)
    E, K, m, d, n = 4, 2, 40, 7168, 2048
    x = synth.randn((m, d), synth.seed_of("wse", m), 1.0).to(torch.bfloat16)
    g = torch.Generator().manual_seed(3)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    w = {}
    for i, (name, a, b) in enumerate((("gate_proj", n, d), ("up_proj", n, d), ("down_proj", d, n))):
        w[name] = synth.quantize_fp8_blocks(synth.randn((a, b), synth.seed_of("wse-w", i), 0.02))
    one = F.expert_ffn(x, w)                     # every expert the same weights, each at its own address
    want = one[:, None].expand(m, K, d)
    st = {k: (q[None].repeat(E, 1, 1).to(DEV), s[None].repeat(E, 1, 1).to(DEV)) for k, (q, s) in w.items()}
    table, _ = ops._stacked_device_table(st, E, d, torch.device(DEV))
    xd, idd, y = x.to(DEV), idx.to(DEV), torch.empty(m, K, d, dtype=torch.bfloat16, device=DEV)
    call = lambda p, b: lib().amla_moe_experts_dev(xd.data_ptr(), m, d, K, idd.data_ptr(), n, E, table.data_ptr(),
                                                   y.data_ptr(), p, b, ops._stream_ptr(xd))
    full, least = lib().amla_moe_experts_dev_workspace_bytes(m, d, K, n, E), _least(call)
    assert least < full
    for b in (full, least, (full + least) // 2):
        y.zero_()
        _run(call, b)
        assert_parity(y, want, f"experts in {b} bytes")


@pytest.mark.parametrize("S,starts,rows", [(5, list(range(28, 54, 2)), 64), (181, [700], 1024), (70, [3, 0, 30], 128)])
def test_prefill_in_the_form_and_parts_that_fit(S, starts, rows):
    """Latent attention where its scratch fits, decompressed where only that does; with and without
    the GEMMs' K parts."""
    B = len(starts)
    print(f"[case] prefill workspace S={S} starts={starts}", flush=True)
    aw = synth.make_layer(CFG, "ws-prefill").attn_weights
    aw = {k: (tuple(t.to(DEV) for t in v) if isinstance(v, tuple) else v.to(DEV)) for k, v in aw.items()}
    hidden = synth.make_hidden(CFG, B, S, f"ws{S}").to(DEV)
    kv = [t.to(DEV) for t in synth.make_kv_cache(CFG, B, rows, starts, f"ws{S}")]
    tab = R.precompute_rope_freqs(CFG, rows).to(DEV)
    want = ops.mla_attention(hidden, aw, tuple(t.clone() for t in kv), starts, tab, CFG)
    out, pos = torch.empty_like(hidden), torch.tensor(starts, dtype=torch.int32, device=DEV)
    freqs = torch.view_as_real(tab).contiguous() if tab.is_complex() else tab
    a = fill_mla_args(hidden, *aw["q_a_proj"], *aw["q_b_proj"], *aw["kv_a_proj_with_mqa"], *aw["kv_b_proj"],
                      *aw["o_proj"], aw["q_a_layernorm"], aw["kv_a_layernorm"], kv[0], kv[1], pos, freqs, None, None,
                      None, out, 0, CFG.rms_norm_eps, ops.softmax_scale(CFG), CFG.num_attention_heads,
                      CFG.qk_nope_head_dim, CFG.v_head_dim)

    def call(p, b):
        a.workspace, a.workspace_bytes = p or hidden.data_ptr(), b
        return lib().amla_mla_prefill(ctypes.byref(a), ops._stream_ptr(hidden))

    full, least = lib().amla_mla_prefill_workspace_bytes(ctypes.byref(a)), _least(call)
    assert least < full
    for b in (full, least, (full + least) // 2):
        out.zero_()
        _run(call, b)
        assert_parity(out, want, f"prefill S={S} in {b} bytes")
