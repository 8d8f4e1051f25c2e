"""Routing and the MoE combine at the sizes where their kernels change: the 64 x 64 logits tiles
(above 64 tokens; K splits, ragged tokens and experts), more than 256 experts, NaN scores, and the
combine's eight-column path against its one-column path."""
import pytest
import torch

from oracle import ref_ffn as F
from amla import ops, synth
from test_gpu_ffn import _cfg, _check_route, _x

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,E,G,TG,K,d", [(64, 256, 8, 4, 8, 256), (65, 256, 8, 4, 8, 256), (127, 40, 4, 2, 3, 96),
                                          (130, 16, 4, 2, 4, 32), (200, 320, 8, 4, 8, 224), (3, 1024, 8, 3, 64, 160)])
def test_route_tiles(m, E, G, TG, K, d):
    print(f"[case] route m={m} E={E} d={d}", flush=True)
    cfg = _cfg(E, G, TG, K)
    h = _x((1, m, d), f"rt{m}{E}")
    gw = synth.randn((E, d), synth.seed_of("rt", E, d), 0.1).to(torch.bfloat16)
    idx, w = ops.route(h.to(DEV), gw.to(DEV), cfg)
    ridx, rw = F.route(h, gw, cfg)
    _check_route(idx, w, ridx, rw, torch.sigmoid(h.float() @ gw.float().T))


def test_route_skips_nan_scores():
    """An expert whose score is NaN is never chosen while others are left."""
    E, d, m = 32, 64, 4
    cfg = _cfg(E, 1, 1, 6)
    h = _x((1, m, d), "rnan").abs() + 0.5
    gw = synth.randn((E, d), synth.seed_of("rnan", E), 0.1).to(torch.bfloat16)
    clean = torch.sigmoid(h.float() @ gw.float().T)
    bad = [0, 7, 31]
    gwn = gw.clone()
    gwn[bad, 3] = float("nan")
    idx, _ = ops.route(h.to(DEV), gwn.to(DEV), cfg)
    clean[..., bad] = -1.0
    assert torch.equal(idx.cpu(), clean.topk(6, dim=-1).indices)


@pytest.mark.parametrize("m,K,d", [(1, 1, 8), (3, 7, 1000), (5, 9, 264), (70, 16, 2056)])
def test_combine_paths_agree_bit_for_bit(m, K, d):
    """Aligned rows (eight columns per thread) against the same rows at a 2-byte offset (one
    column per thread) and the reference's roundings."""
    print(f"[case] combine m={m} K={K} d={d}", flush=True)
    sh, eo = _x((m, d), f"c8s{d}"), _x((m, K, d), f"c8e{d}")
    w = torch.rand(m, K, generator=torch.Generator().manual_seed(d))
    routed = torch.zeros(m, d, dtype=torch.bfloat16)
    for k in range(K):
        routed += w[:, k, None].to(torch.bfloat16) * eo[:, k]
    want = sh + routed * 2.5
    for off in (0, 1):
        def place(t):
            buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)
            v = buf[off:off + t.numel()].view(t.shape)
            v.copy_(t)
            return v
        shd, eod, out, wd = place(sh), place(eo), place(torch.zeros(m, d, dtype=torch.bfloat16)), w.to(DEV)
        ops.check(ops.lib().amla_moe_combine(shd.data_ptr(), eod.data_ptr(), wd.data_ptr(), m, K, d, 2.5,
                                             out.data_ptr(), ops._stream_ptr(shd)), "moe_combine")
        assert torch.equal(out.cpu(), want), off
