"""The calls a serving loop for DeepSeek-R1 makes of this package, as measured cases.

One layer's attention half (decode and prefill, over short and long caches, one sequence and
many), the FFN of the dense layers, the MoE block, the output head and the sampler, each
through the public function an engine calls.  Sizes are the R1 configuration
(``amla.config.DeepSeekConfig``); batch, prompt and context lengths span what one GPU serves.

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same ranges,
``prepare`` what the engine holds before the call, ``run`` one call, ``work`` the bytes and
operations the call cannot do without, ``tolerance`` the difference another correct
implementation at the same precision may show, and ``exact`` the result in 64 bits.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deepseek-on-one-gpu_amd"))

from amla import ops  # noqa: E402
from amla.config import DeepSeekConfig  # noqa: E402

CFG = DeepSeekConfig()
DEV = "cuda"
BF16, F32, F64, FP8 = torch.bfloat16, torch.float32, torch.float64, torch.float8_e4m3fn
H, NOPE, ROPE, VD = CFG.num_attention_heads, CFG.qk_nope_head_dim, CFG.qk_rope_head_dim, CFG.v_head_dim
LORA, QLORA, D = CFG.kv_lora_rank, CFG.q_lora_rank, CFG.hidden_size
E, TOPK, EI = CFG.n_routed_experts, CFG.num_experts_per_tok, CFG.moe_intermediate_size
PROJ = {
    "q_a_proj": (QLORA, D),
    "q_b_proj": (H * (NOPE + ROPE), QLORA),
    "kv_a_proj_with_mqa": (LORA + ROPE, D),
    "kv_b_proj": (H * (NOPE + VD), LORA),
    "o_proj": (D, H * VD),
}
MAX_PREFILL, MAX_TOKENS, MAX_MOE = 4096, 2048, 2000
MAX_DECODE_ROWS, MAX_PAST = 8 * 32768, 32767


# ------------------------------------------------------------------ the cases

def _mla(entry, batch, new, past_lo, past_hi):
    return {"kind": "mla", "entry": entry, "batch": batch, "new": new, "past_lo": past_lo, "past_hi": past_hi}


def listed():
    return [
        # one user, a chat turn just begun: the smallest step, launches and latency count
        {"name": "decode_b1_short", **_mla("layer", 1, 1, 256, 256)},
        # eight users deep in 32k contexts: the repository's headline step
        {"name": "decode_b8_32k", **_mla("layer", 8, 1, 32767, 32767)},
        # thirty-two users at mixed contexts between 1k and 16k (continuous batching)
        {"name": "decode_b32_ragged", **_mla("attention", 32, 1, 1024, 16383)},
        # a first prompt of a few paragraphs
        {"name": "prefill_333", **_mla("attention", 1, 333, 0, 0)},
        # a 4k prompt, or one chunk of a longer one
        {"name": "prefill_4096", **_mla("layer", 1, 4096, 0, 0)},
        # the next user message of a running chat: a few dozen new tokens over an 8k cache
        {"name": "followup_50_8k", **_mla("layer", 1, 50, 8100, 8100)},
        # FFN of the three dense layers: a decode step of eight, and a prompt
        {"name": "dense_ffn_8", "kind": "dense", "tokens": 8},
        {"name": "dense_ffn_1000", "kind": "dense", "tokens": 1000},
        # FFN of the 58 MoE layers, experts resident: a decode step of eight, and a prompt
        {"name": "moe_8", "kind": "moe", "tokens": 8},
        {"name": "moe_2000", "kind": "moe", "tokens": MAX_MOE},
        # logits of the last tokens of eight sequences, and drawing their next tokens
        {"name": "head_8", "kind": "head", "rows": 8},
        {"name": "sample_8", "kind": "sample", "rows": 8, "temperature": 0.6, "top_p": 0.95},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(["decode", "decode", "prefill", "followup", "dense", "moe", "moe", "head", "sample"])
    entry = rng.choice(["layer", "attention"])
    if what == "decode":
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 16, min(MAX_PAST, MAX_DECODE_ROWS // batch - 1))
        lo = hi if rng.random() < 0.4 else _log_int(rng, max(1, hi // 16), hi)
        return _mla(entry, batch, 1, lo, hi)
    if what == "prefill":
        return _mla(entry, 1, _log_int(rng, 2, MAX_PREFILL), 0, 0)
    if what == "followup":
        new = _log_int(rng, 2, 1024)
        past = _log_int(rng, 256, 12000)
        return _mla(entry, 1, new, past, past)
    if what == "dense":
        return {"kind": "dense", "tokens": _log_int(rng, 1, MAX_TOKENS)}
    if what == "moe":
        return {"kind": "moe", "tokens": _log_int(rng, 1, MAX_MOE)}
    if what == "head":
        return {"kind": "head", "rows": _log_int(rng, 1, 64)}
    return {"kind": "sample", "rows": _log_int(rng, 1, 64), "temperature": rng.choice([0.0, 0.6, 1.0]),
            "top_p": rng.choice([0.8, 0.9, 0.95])}


def _past(case):
    """Cached rows of each sequence: spread evenly over [past_lo, past_hi], in no order."""
    lo, hi, n = case["past_lo"], case["past_hi"], case["batch"]
    return [lo + int((hi - lo) * ((i * 0.6180339887498949 + 0.37) % 1.0)) for i in range(n)]


# ------------------------------------------------------------------ inputs

class _Draw:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def randn(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=F32)
        return t.mul_(std) if std != 1.0 else t

    def bf16(self, *shape, std=1.0):
        return self.randn(*shape, std=std).to(BF16)

    def gamma(self, n):
        return (1.0 + self.randn(n, std=0.1)).to(BF16)

    def fp8(self, n, k, std=0.02):
        """N(0, std) weights quantised per 128 x 128 block (scale_inv = amax / 448), as the checkpoint holds them."""
        nb, kb = -(-n // 128), -(-k // 128)
        w = torch.zeros(nb * 128, kb * 128, device=DEV)
        w[:n, :k] = self.randn(n, k, std=std)
        blocks = w.view(nb, 128, kb, 128)
        scale = (blocks.abs().amax(dim=(1, 3)) / 448.0).clamp_min(1e-12)
        q = (blocks / scale[:, None, :, None]).clamp_(-448.0, 448.0).view(nb * 128, kb * 128)[:n, :k]
        return q.to(FP8).contiguous(), scale.contiguous()

    def experts(self, n, k, count):
        """`count` stacked (n, k) weights of the MoE layer."""
        w = torch.empty(count, n, k, dtype=FP8, device=DEV)
        s = torch.empty(count, n // 128, k // 128, device=DEV)
        step = 16
        for e in range(0, count, step):
            c = min(step, count - e)
            q, sc = self.fp8(c * n, k)
            w[e:e + c] = q.view(c, n, k)
            s[e:e + c] = sc.view(c, n // 128, k // 128)
        return w, s


def prepare(case, seed):
    r = _Draw(seed)
    kind = case["kind"]
    if kind == "mla":
        B, S, past = case["batch"], case["new"], _past(case)
        rows = -(-(max(past) + S) // 256) * 256
        aw = {name: r.fp8(n, k) for name, (n, k) in PROJ.items()}
        aw["q_a_layernorm"], aw["kv_a_layernorm"] = r.gamma(QLORA), r.gamma(LORA)
        ckv = torch.zeros(B, rows, LORA, dtype=BF16, device=DEV)
        kpe = torch.zeros(B, rows, ROPE, dtype=BF16, device=DEV)
        for b, p in enumerate(past):
            ckv[b, :p] = r.bf16(p, LORA)
            kpe[b, :p] = r.bf16(p, ROPE)
        st = {"aw": aw, "gamma_in": r.gamma(D), "cache": (ckv, kpe), "hidden": r.bf16(B, S, D),
              "rope": ops.precompute_rope_freqs(CFG, rows, DEV), "max_context": max(past) + S}
        # a decode loop keeps its positions on the device; a prompt starts at one known position
        st["position"] = torch.tensor(past, dtype=torch.int32, device=DEV) if S == 1 else past[0]
    elif kind == "dense":
        I = CFG.intermediate_size
        st = {"hidden": r.bf16(1, case["tokens"], D), "mlp": {"gate_proj": r.fp8(I, D), "up_proj": r.fp8(I, D),
                                                              "down_proj": r.fp8(D, I)}}
    elif kind == "moe":
        st = {"hidden": r.bf16(1, case["tokens"], D), "gate": r.bf16(E, D, std=0.02),
              "shared": {"gate_proj": r.fp8(EI, D), "up_proj": r.fp8(EI, D), "down_proj": r.fp8(D, EI)},
              "experts": {"gate_proj": r.experts(EI, D, E), "up_proj": r.experts(EI, D, E),
                          "down_proj": r.experts(D, EI, E)}}
    elif kind == "head":
        st = {"hidden": r.bf16(case["rows"], 1, D, std=2.0), "norm": r.gamma(D),
              "lm_head": torch.cat([r.bf16(CFG.vocab_size // 8, D, std=0.02) for _ in range(8)])}
    else:
        # a model's logits: a broad bulk and a few dozen likely tokens per row
        lg = r.randn(case["rows"], CFG.vocab_size, std=2.0)
        pos = torch.randint(CFG.vocab_size, (case["rows"], 40), generator=r.g, device=DEV)
        lg.scatter_(1, pos, 12.0 + r.randn(case["rows"], 40, std=2.0))
        st = {"logits": lg, "draw_seed": seed * 7919 + 1}
    st["case"] = case
    return st


# ------------------------------------------------------------------ one call

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "mla":
        kw = {"max_context": st["max_context"]} if case["new"] == 1 else {}
        if case["entry"] == "layer":
            out = ops.mla_layer(st["hidden"], st["gamma_in"], st["aw"], st["cache"], st["position"], st["rope"], CFG, **kw)
        else:
            out = ops.mla_attention(st["hidden"], st["aw"], st["cache"], st["position"], st["rope"], CFG, **kw)
        return (out, *st["cache"])
    if kind == "dense":
        return ops.dense_ffn(st["hidden"], st["mlp"])
    if kind == "moe":
        return ops.moe_block(st["hidden"], st["gate"], st["shared"], st["experts"], CFG)
    if kind == "head":
        return ops.final_logits(st["hidden"], st["norm"], st["lm_head"], CFG)
    return ops.sample(st["logits"], case["temperature"], case["top_p"], seed=st["draw_seed"])


# ------------------------------------------------------------------ what it cannot do without

def _weights(n, k):
    return n * k + 4 * -(-n // 128) * -(-k // 128)


def work(case):
    kind = case["kind"]
    if kind == "mla":
        B, S, past = case["batch"], case["new"], _past(case)
        w = sum(_weights(n, k) for n, k in PROJ.values()) + 2 * (QLORA + LORA + (D if case["entry"] == "layer" else 0))
        rows = sum(past)
        byts = w + (rows + B * S) * 2 * (LORA + ROPE) + 4 * B * S * D + 4 * ROPE * (max(past) + S)
        proj = 2 * sum(n * k for name, (n, k) in PROJ.items() if name != "kv_b_proj")
        pairs = sum(S * p + S * (S + 1) // 2 for p in past)
        # the cheaper of the two forms of the attention: kv_b applied to the query and the
        # output of every new token, or to every cached row
        kvb = 2 * PROJ["kv_b_proj"][0] * LORA
        absorbed = B * S * kvb + pairs * 2 * H * (2 * LORA + ROPE)
        direct = (rows + B * S) * kvb + pairs * 2 * H * (NOPE + ROPE + VD)
        return {"bytes": byts, "flops": B * S * proj + min(absorbed, direct)}
    if kind == "dense":
        M, I = case["tokens"], CFG.intermediate_size
        return {"bytes": 2 * _weights(I, D) + _weights(D, I) + 4 * M * D, "flops": 6 * M * D * I}
    if kind == "moe":
        M = case["tokens"]
        # experts that get a token when the choices fall evenly
        used = E * (1.0 - (1.0 - TOPK / E) ** M)
        one = 2 * _weights(EI, D) + _weights(D, EI)
        return {"bytes": int((used + 1) * one) + 2 * E * D + 4 * M * D,
                "flops": 6 * M * (TOPK + 1) * D * EI + 2 * M * E * D}
    if kind == "head":
        M, V = case["rows"], CFG.vocab_size
        return {"bytes": 2 * V * D + 2 * D + 2 * M * D + 4 * M * V, "flops": 2 * M * V * D}
    return {"bytes": 4 * case["rows"] * CFG.vocab_size + 8 * case["rows"], "flops": 4 * case["rows"] * CFG.vocab_size}


def tolerance(case):
    """About four times the distance from `exact` measured at the sizes above."""
    kind = case["kind"]
    if kind == "mla":
        # attention alone 0.0038-0.0058 (bf16 operands of six products in a row); with the
        # residual, which dwarfs it, 0.0017-0.0018 (one bf16 rounding); new cache rows 0.0029
        return {"rel": 8e-3 if case["entry"] == "layer" else 2.4e-2}
    if kind == "dense":
        return {"rel": 1.6e-2}  # 0.0039
    if kind == "moe":
        return {"rel": 2.2e-2}  # 0.0053
    if kind == "head":
        return {"rel": 1e-2}  # 0.0025, the norm's bf16 output
    return "exact"


# ------------------------------------------------------------------ 64 bits

def _deq(pair):
    w, s = pair
    n, k = w.shape
    out = w.to(F64)
    for j in range(s.shape[1]):
        out[:, 128 * j:128 * (j + 1)] *= s[:, j].to(F64).repeat_interleave(128)[:n, None]
    return out


def _norm(x, gamma):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + CFG.rms_norm_eps) * gamma.to(F64)


def _rotate(x, f):
    """x (rows, .., 64) by f (rows, 32) complex, pairs (2i, 2i + 1)."""
    z = torch.view_as_complex(x.reshape(*x.shape[:-1], ROPE // 2, 2).contiguous())
    f = f.view(f.shape[0], *([1] * (z.dim() - 2)), ROPE // 2)
    return torch.view_as_real(z * f).flatten(-2)


def _swiglu(x, w):
    g = x @ _deq(w["gate_proj"]).T
    return (g * torch.sigmoid(g) * (x @ _deq(w["up_proj"]).T)) @ _deq(w["down_proj"]).T


def _exact_mla(case, st):
    aw, (ckv, kpe) = st["aw"], st["cache"]
    B, S = case["batch"], case["new"]
    hid = st["hidden"].to(F64).view(B * S, D)
    x = _norm(hid, st["gamma_in"]) if case["entry"] == "layer" else hid
    q = (_norm(x @ _deq(aw["q_a_proj"]).T, aw["q_a_layernorm"]) @ _deq(aw["q_b_proj"]).T).view(B, S, H, NOPE + ROPE)
    new = (x @ _deq(aw["kv_a_proj_with_mqa"]).T).view(B, S, LORA + ROPE)
    kvb = _deq(aw["kv_b_proj"]).view(H, NOPE + VD, LORA)
    mscale = 0.1 * CFG.rope_scaling_mscale_all_dim * math.log(CFG.rope_scaling_factor) + 1.0
    scale = mscale / math.sqrt(NOPE + ROPE)
    freqs = st["rope"].to(torch.complex128)
    ckv, kpe = ckv.to(F64), kpe.to(F64)
    heads = torch.empty(B * S, H * VD, dtype=F64, device=DEV)
    for b, p in enumerate(_past(case)):
        T = p + S
        ckv[b, p:T], kpe[b, p:T] = new[b, :, :LORA], new[b, :, LORA:]
        c, kr = _norm(ckv[b, :T], aw["kv_a_layernorm"]), _rotate(kpe[b, :T], freqs[:T])
        keys = torch.cat([c, kr], dim=1)
        qp = _rotate(q[b, :, :, NOPE:], freqs[p:T])
        late = torch.arange(T, device=DEV)[None, :] > torch.arange(p, T, device=DEV)[:, None]
        step = max(1, min(H, (1 << 27) // (S * T)))
        for h0 in range(0, H, step):
            hs = range(h0, min(H, h0 + step))
            qa = torch.stack([torch.cat([q[b, :, h, :NOPE] @ kvb[h, :NOPE], qp[:, h]], dim=1) for h in hs])
            sc = (qa.reshape(-1, LORA + ROPE) @ keys.T).view(len(hs), S, T) * scale
            pr = torch.softmax(sc.masked_fill_(late, -math.inf), dim=-1)
            lat = (pr.view(-1, T) @ c).view(len(hs), S, LORA)
            for i, h in enumerate(hs):
                heads[b * S:(b + 1) * S, h * VD:(h + 1) * VD] = lat[i] @ kvb[h, NOPE:].T
    out = heads @ _deq(aw["o_proj"]).T
    if case["entry"] == "layer":
        out = out + hid
    return out.view(B, S, D), ckv, kpe


def _exact_moe(case, st):
    x = st["hidden"].to(F64).view(-1, D)
    M = x.shape[0]
    sc = torch.sigmoid(x @ st["gate"].to(F64).T)
    top_g = sc.view(M, CFG.n_group, -1).amax(-1).topk(CFG.topk_group, dim=-1).indices
    keep = torch.zeros(M, CFG.n_group, dtype=torch.bool, device=DEV).scatter_(1, top_g, True)
    masked = sc * keep.repeat_interleave(E // CFG.n_group, dim=1)
    w, idx = masked.topk(TOPK, dim=-1)
    w = w / (w.sum(-1, keepdim=True) + 1e-9)
    routed = torch.zeros(M, D, dtype=F64, device=DEV)
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            one = {name: (st["experts"][name][0][e], st["experts"][name][1][e]) for name in st["experts"]}
            routed.index_add_(0, t, w[t, k, None] * _swiglu(x[t], one))
    return (_swiglu(x, st["shared"]) + routed * CFG.routed_scaling_factor).view(1, M, D)


def exact(case, seed):
    if case["kind"] == "sample":
        return None  # tokens
    st = prepare(case, seed)
    if case["kind"] == "mla":
        return _exact_mla(case, st)
    if case["kind"] == "dense":
        return _swiglu(st["hidden"].to(F64).view(-1, D), st["mlp"]).view(1, -1, D)
    if case["kind"] == "moe":
        return _exact_moe(case, st)
    x = _norm(st["hidden"].to(F64).view(-1, D), st["norm"])
    w = st["lm_head"]
    return torch.cat([x @ w[v:v + 16160].to(F64).T for v in range(0, w.shape[0], 16160)], dim=1).view(-1, 1, w.shape[0])
