"""Prefill of a few new tokens over a filled cache, where the attention runs in latent space: one
token and many, several sequences with their own start, more tokens than one launch holds, tile
and split edges, chosen and not; against the oracle per sequence (its roundings), per head and
after o_proj, with the cache rows written."""
import pytest
import torch

from oracle import ref_ops as R
from amla import ops, synth
from amla.config import DeepSeekConfig
from _prefill import runs_latent
from _tol import assert_bf16_ulps, assert_heads_parity, assert_parity

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CFG = DeepSeekConfig()


@pytest.fixture(scope="module")
def layer():
    return synth.make_layer(CFG, "latent-prefill")


def _gpu(aw):
    return {k: (tuple(t.to(DEV) for t in v) if isinstance(v, tuple) else v.to(DEV)) for k, v in aw.items()}


@pytest.mark.parametrize("S,starts", [(2, [1023]), (7, [640]), (33, [1500]), (65, [1951]), (9, [513, 0, 1200, 70]),
                                      (40, [900, 31]), (5, list(range(28, 54, 2)))])
def test_new_tokens_over_a_cache(layer, S, starts):
    print(f"[case] latent prefill S={S} starts={starts}", flush=True)
    B = len(starts)
    rows = max(starts) + S + 5
    assert runs_latent(B, S, rows)
    hidden = synth.make_hidden(CFG, B, S, f"lp{S}")
    ckv, kpe = synth.make_kv_cache(CFG, B, rows, starts, f"lp{S}")
    tab = R.precompute_rope_freqs(CFG, rows)
    cref, kref = ckv.clone(), kpe.clone()
    want_h, want = R.mla_attention_per_sequence_parts(hidden, layer.attn_weights, (cref, kref), starts, tab, CFG)
    cd, kd = ckv.to(DEV), kpe.to(DEV)
    heads = torch.empty(B, S, CFG.num_attention_heads * CFG.v_head_dim, dtype=torch.bfloat16, device=DEV)
    got = ops.mla_attention(hidden.to(DEV), _gpu(layer.attn_weights), (cd, kd), starts, tab.to(DEV), CFG, attn_out=heads)
    torch.cuda.synchronize()
    assert_heads_parity(heads, want_h, CFG.num_attention_heads, f"latent prefill S={S} heads")
    assert_parity(got, want, f"latent prefill S={S}")
    for b, p in enumerate(starts):
        assert_bf16_ulps(cd[b, p:p + S], cref[b, p:p + S], 2, "new latent rows")
        assert_bf16_ulps(kd[b, p:p + S], kref[b, p:p + S], 2, "new rope rows")
        assert torch.equal(cd[b, :p].cpu(), ckv[b, :p]) and torch.equal(cd[b, p + S:].cpu(), ckv[b, p + S:])


def test_prompt_and_token_by_token_agree(layer):
    """The same 12 new tokens at once (latent attention over 1024 + 12 rows) and one decode step
    each: the same rows in the cache and the same outputs to the bf16 bar."""
    S, p, rows = 12, 1024, 1100
    aw = _gpu(layer.attn_weights)
    hidden = synth.make_hidden(CFG, 1, S, "lp-step").to(DEV)
    ckv, kpe = (t.to(DEV) for t in synth.make_kv_cache(CFG, 1, rows, p, "lp-step"))
    tab = R.precompute_rope_freqs(CFG, rows).to(DEV)
    c2, k2 = ckv.clone(), kpe.clone()
    at_once = ops.mla_attention(hidden, aw, (ckv, kpe), p, tab, CFG)
    steps = torch.cat([ops.mla_attention(hidden[:, i:i + 1], aw, (c2, k2), p + i, tab, CFG) for i in range(S)], dim=1)
    torch.cuda.synchronize()
    assert_parity(at_once, steps, "prompt vs token by token")
    assert_bf16_ulps(ckv, c2, 2, "cache rows")


@pytest.mark.parametrize("S,starts,latent", [(5, [700], True), (66, [3, 0, 30], False), (130, [1], False)])
def test_norm_weights_at_any_alignment(layer, S, starts, latent):
    """The row passes between the projections and the latent merge read the norm weights 16 bytes at
    a time where these are aligned: weights two bytes off give the same result."""
    print(f"[case] prefill norm weights S={S} starts={starts}", flush=True)
    B, rows = len(starts), max(starts) + S + 2
    assert runs_latent(B, S, rows) == latent
    aw = _gpu(layer.attn_weights)
    hidden = synth.make_hidden(CFG, B, S, "lp-gamma").to(DEV)
    kv = [t.to(DEV) for t in synth.make_kv_cache(CFG, B, rows, starts, "lp-gamma")]
    tab = R.precompute_rope_freqs(CFG, rows).to(DEV)

    def off(g):
        buf = torch.empty(g.numel() + 1, dtype=g.dtype, device=DEV)
        buf[1:] = g
        return buf[1:]

    c2, c3 = [t.clone() for t in kv], [t.clone() for t in kv]
    want = ops.mla_attention(hidden, aw, tuple(kv), starts, tab, CFG)
    got = ops.mla_attention(hidden, dict(aw, kv_a_layernorm=off(aw["kv_a_layernorm"])), tuple(c2), starts, tab, CFG)
    both = ops.mla_attention(hidden, dict(aw, kv_a_layernorm=off(aw["kv_a_layernorm"]),
                                          q_a_layernorm=off(aw["q_a_layernorm"])), tuple(c3), starts, tab, CFG)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(kv, c2))
    # the q_a norm sums an unaligned row in another order
    assert_parity(both, want, f"both weights off S={S}")


@pytest.mark.parametrize("S,p", [(12, 1500), (70, 4000)])
def test_heads_lose_nothing_to_16_bit_sums(layer, S, p):
    """Rows about one latent vector under equal scores, where the roundings of a split's sums and of
    the merged latent do not average out: the heads against 64 bits.  Left are their own rounding to
    bf16 (taken from the 64-bit values) and the one of p r_t, 2^-9 at most on each weight and, the
    row norms spread over several bf16 steps, under 2^-11 on a sum of them."""
    T = p + S
    assert runs_latent(1, S, T)
    print(f"[case] latent prefill precision S={S} T={T}", flush=True)
    aw = _gpu(layer.attn_weights)
    aw["q_b_proj"] = (aw["q_b_proj"][0], aw["q_b_proj"][1] * 1e-12)
    hidden = synth.make_hidden(CFG, 1, S, "lp-flat").to(DEV)
    g = torch.Generator().manual_seed(S)
    ckv = (torch.randn(1, 1, 512, generator=g) + 0.5 * torch.randn(1, T, 512, generator=g)).to(torch.bfloat16).to(DEV)
    kpe = torch.randn(1, T, 64, generator=g).to(torch.bfloat16).to(DEV)
    tab = R.precompute_rope_freqs(CFG, T).to(DEV)
    heads = torch.empty(1, S, 128 * 128, dtype=torch.bfloat16, device=DEV)
    ops.mla_attention(hidden, aw, (ckv, kpe), p, tab, CFG, attn_out=heads)
    torch.cuda.synchronize()
    c = ckv[0].double().cpu()
    c = c * torch.rsqrt(c.pow(2).mean(1, keepdim=True) + CFG.rms_norm_eps) * layer.attn_weights["kv_a_layernorm"].double()
    lat = (c.cumsum(0) / torch.arange(1, T + 1, dtype=torch.float64)[:, None])[p:]
    w, s = layer.attn_weights["kv_b_proj"]
    w = (w.double() * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)).view(128, 256, 512)[:, 128:]
    want = torch.einsum("sl,hvl->shv", lat, w).reshape(S, 128 * 128)
    n = want.norm()
    err, own = (heads[0].double().cpu() - want).norm() / n, (want.to(torch.bfloat16).double() - want).norm() / n
    print(f"    error {err:.6f}, rounding of the result {own:.6f}", flush=True)
    assert err ** 2 <= own ** 2 + 2.0 ** -22
