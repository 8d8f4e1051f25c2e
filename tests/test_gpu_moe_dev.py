"""amla_moe_experts_dev (the routed experts of moe_block grouped on the device) against the
oracle's expert_ffn of every (token, k) slot, and moe_block captured in a HIP graph.

The reference brings the chosen indices to the host before its expert loop
(gpu_transfer.py:60, forward.py:139-151); the device schedule replaces that step, so the
results are checked against the same oracle as amla_moe_experts: per slot,
expert_ffn(hidden[token], experts[index]) (oracle/ref_ffn.py), to the bf16 bar of _tol."""
import pytest
import torch

from oracle import ref_ffn as F
from amla import ops, synth
from _tol import assert_parity
from test_gpu_ffn import _cfg, _dev, _mlp, _x

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SENTINEL = 0x7E11   # bf16 bit pattern of rows the call must not write


def _stacked(table, E):
    return {k: (torch.stack([table[e][k][0] for e in range(E)]).to(DEV),
                torch.stack([table[e][k][1] for e in range(E)]).to(DEV)) for k in ("gate_proj", "up_proj", "down_proj")}


def _run_dev(h, idx, stacked, E, n_inter, null_experts=()):
    """amla_moe_experts_dev through the C-ABI; returns (expert_out, header ints)."""
    m, K = idx.shape
    d = h.shape[1]
    table, _ = ops._stacked_device_table(stacked, E, d, torch.device(DEV))
    if null_experts:
        table = table.clone().view(6, E)
        for e in null_experts:
            table[:, e] = 0
        table = table.view(-1)
    hd = h.to(DEV)
    eout = torch.full((m, K, d), SENTINEL, dtype=torch.int16, device=DEV).view(torch.bfloat16)
    need = ops.lib().amla_moe_experts_dev_workspace_bytes(m, d, K, n_inter, E)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    idx_d = idx.to(torch.int64).contiguous().to(DEV)
    ops.check(ops.lib().amla_moe_experts_dev(hd.data_ptr(), m, d, K, idx_d.data_ptr(), n_inter, E, table.data_ptr(),
                                             eout.data_ptr(), ws.data_ptr(), need, ops._stream_ptr(hd)),
              "moe_experts_dev")
    torch.cuda.synchronize()
    return eout.cpu(), ws[:16].view(torch.int32).cpu().tolist()


def _want(h, idx, table, skip=lambda e: False):
    m, K = idx.shape
    want = torch.empty(m, K, h.shape[1], dtype=torch.bfloat16)
    for e in sorted(set(idx.flatten().tolist())):
        if e < 0 or e not in table or skip(e):
            continue
        sel = (idx == e).nonzero()
        want[sel[:, 0], sel[:, 1]] = F.expert_ffn(h[sel[:, 0]], table[e])
    return want


@pytest.mark.parametrize("E,K,m,dup", [(256, 8, 8, False), (6, 3, 150, False), (16, 8, 200, False),
                                       (2, 1, 300, False), (8, 4, 5, True), (1, 4, 1, True),
                                       (4, 2, 40, False), (12, 3, 60, False)])
def test_moe_experts_dev_vs_expert_ffn(E, K, m, dup):
    """Groups on the skinny GEMM (up to 32 tokens), on the tiles (more) and made larger than m by
    repeated indices; the header's counts: groups of at most min(m, 64) slots, 256-row units of the
    larger ones."""
    print(f"[case] moe_experts_dev E={E} K={K} m={m} dup={dup}", flush=True)
    d, i = 256, 256
    h = _x((m, d), f"mdev{E}{K}{m}")
    g = torch.Generator().manual_seed(E * 7919 + K * 31 + m)
    if dup:
        idx = torch.randint(0, E, (m, K), generator=g)
    else:
        idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    table = {e: _mlp(d, i, f"mdev-expert{e}") for e in range(E)}
    got, hdr = _run_dev(h, idx, _stacked(table, E), E, i)
    assert hdr[0] == m * K and hdr[3] == 0
    counts = torch.bincount(idx.flatten(), minlength=E)
    sb = min(m, 64)
    assert hdr[1] == int(((counts >= 1) & (counts <= sb)).sum())
    assert hdr[2] == int(((counts + 255) // 256 * (counts > sb)).sum())
    assert_parity(got, _want(h, idx, table), f"moe_experts_dev E={E} K={K} m={m}")


def test_moe_experts_dev_skips_and_counts():
    """Negative indices are left out silently; indices >= E and experts with a NULL table entry
    are left out and counted; their rows keep what they held."""
    print("[case] moe_experts_dev skipped slots", flush=True)
    E, K, m, d, i = 12, 4, 40, 256, 256
    h = _x((m, d), "mdev-skip")
    g = torch.Generator().manual_seed(4242)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    idx[::7, 0] = -1
    idx[3::11, 1] = E + 2
    null = (5,)
    table = {e: _mlp(d, i, f"mdev-skip{e}") for e in range(E)}
    got, hdr = _run_dev(h, idx, _stacked(table, E), E, i, null_experts=null)
    skipped = (idx >= E) | (idx == 5)
    left = idx < 0
    assert hdr[3] == int(skipped.sum())
    assert hdr[0] == m * K - int(skipped.sum()) - int(left.sum())
    untouched = got.view(torch.int16)[skipped | left]
    assert (untouched == SENTINEL).all()
    keep = ~(skipped | left)
    want = _want(h, idx, table, skip=lambda e: e in null)
    assert_parity(got[keep], want[keep], "moe_experts_dev with skipped slots")


@pytest.mark.parametrize("m", [8, 40])
def test_moe_experts_dev_r1_expert_shape(m):
    """Decode-sized batches at the R1 expert shape (hidden 7168, intermediate 2048): the K-part
    sums of the skinny path at full size, in entries of at most 16 rows (m = 8) and of 32 (m = 40:
    each of the 4 experts gets about 20 rows)."""
    print(f"[case] moe_experts_dev R1 shape m={m} K=2 E=4", flush=True)
    E, K, d, i = 4, 2, 7168, 2048
    h = _x((m, d), f"mdev-r1-{m}")
    g = torch.Generator().manual_seed(77 + m)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    counts = torch.bincount(idx.flatten(), minlength=E)
    if m > 16:
        assert int(counts.min()) > 16, "every group should be longer than 16 rows"
    table = {e: _mlp(d, i, f"mdev-r1-{e}") for e in range(E)}
    got, hdr = _run_dev(h, idx, _stacked(table, E), E, i)
    assert hdr[0] == m * K and hdr[3] == 0
    assert_parity(got, _want(h, idx, table), f"moe_experts_dev R1 shape m={m}")


def test_moe_block_batch64_r1_shape_device_and_host_grouping_agree():
    """moe_block at batch 64 with R1-shaped experts (16 stacked experts, 8 per token): device
    grouping (groups of up to about 40 rows) against host grouping, and the device path's expert
    outputs against the oracle's expert_ffn per slot."""
    print("[case] moe_block batch 64 R1 expert shape, device vs host grouping", flush=True)
    E, K, m, d, i = 16, 8, 64, 7168, 2048
    cfg = _cfg(E, 4, 2, K)
    h = _x((m, 1, d), "mdev-b64")
    gw = synth.randn((E, d), synth.seed_of("mdev-b64-router", E), 0.02).to(torch.bfloat16)
    shared = _mlp(d, i, "mdev-b64-shared")
    table = {e: _mlp(d, i, f"mdev-b64-{e}") for e in range(E)}
    stacked = _stacked(table, E)
    hd, gwd, shd = h.to(DEV), gw.to(DEV), _dev(shared)
    dev_got = ops.moe_block(hd, gwd, shd, stacked, cfg)
    host_got = ops.moe_block(hd, gwd, shd, stacked, cfg, device_grouping=False)
    idx, _ = ops.route(hd, gwd, cfg)
    torch.cuda.synchronize()
    idx = idx.reshape(m, K).cpu()
    counts = torch.bincount(idx.flatten(), minlength=E)
    assert int(counts.max()) > 16, "some group should be longer than 16 rows"
    assert_parity(dev_got, host_got, "moe_block batch 64: device vs host grouping")
    got, hdr = _run_dev(h.reshape(m, d), idx, stacked, E, i)
    assert hdr[0] == m * K and hdr[3] == 0
    assert_parity(got, _want(h.reshape(m, d), idx, table), "moe_experts_dev batch 64 R1 shape")


def test_device_table_not_reused_for_new_tensors_at_the_same_addresses():
    """Two stacked expert sets in a row with the same E but a different intermediate size; the
    first is freed before the second is made, so the allocator may hand out the same base
    addresses: the second call must get its own pointer table (right per-expert steps)."""
    print("[case] stacked device table keyed by shapes", flush=True)
    E, K, m, d = 4, 2, 6, 256
    h = _x((m, d), "mdev-key")
    g = torch.Generator().manual_seed(5)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    for i in (256, 512):
        table = {e: _mlp(d, i, f"mdev-key-{i}-{e}") for e in range(E)}
        stacked = _stacked(table, E)
        got, hdr = _run_dev(h, idx, stacked, E, i)
        assert hdr[0] == m * K and hdr[3] == 0
        assert_parity(got, _want(h, idx, table), f"moe_experts_dev n_inter={i}")
        dtab, n_inter = ops._stacked_device_table(stacked, E, d, torch.device(DEV))
        step = stacked["gate_proj"][0][0].numel()
        assert n_inter == i
        assert int(dtab[1]) - int(dtab[0]) == step
        del stacked, table, dtab
        torch.cuda.synchronize()
        torch.cuda.empty_cache()


def test_moe_block_device_and_host_grouping_agree_with_the_oracle():
    print("[case] moe_block device vs host grouping", flush=True)
    E, d, i = 64, 256, 256
    cfg = _cfg(E, 8, 4, 6)
    h = _x((4, 3, d), "mdev-block")
    gw = synth.randn((E, d), synth.seed_of("mdev-router", E), 0.1).to(torch.bfloat16)
    shared = _mlp(d, i, "mdev-shared")
    table = {e: _mlp(d, i, f"mdev-b{e}") for e in range(E)}
    stacked = _stacked(table, E)
    dev_got = ops.moe_block(h.to(DEV), gw.to(DEV), _dev(shared), stacked, cfg)
    host_got = ops.moe_block(h.to(DEV), gw.to(DEV), _dev(shared), stacked, cfg, device_grouping=False)
    torch.cuda.synchronize()
    want = F.moe_block(h, gw, shared, lambda e: table[e], cfg)
    assert_parity(dev_got, want, "moe_block device grouping")
    assert_parity(host_got, want, "moe_block host grouping")


def test_moe_block_in_a_hip_graph():
    """route + shared expert + device-grouped experts + combine captured once, replayed on
    new inputs (so the routing changes), with eager work between replays: each replay equals
    the eager call on the same input, and the first also the oracle."""
    print("[case] moe_block graph capture E=32 K=4 B=6", flush=True)
    E, d, i = 32, 256, 256
    cfg = _cfg(E, 4, 2, 4)
    gw = synth.randn((E, d), synth.seed_of("mdev-graph-router", E), 0.1).to(torch.bfloat16)
    shared = _mlp(d, i, "mdev-graph-shared")
    table = {e: _mlp(d, i, f"mdev-g{e}") for e in range(E)}
    stacked = _stacked(table, E)
    gwd, shd = gw.to(DEV), _dev(shared)
    inputs = [_x((6, 1, d), f"mdev-graph-{r}") for r in range(4)]
    static_h = inputs[0].to(DEV)
    ops.moe_block(static_h, gwd, shd, stacked, cfg)            # warm-up: tables, workspaces
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_out = ops.moe_block(static_h, gwd, shd, stacked, cfg)
    routes = set()
    for r, x in enumerate(inputs):
        static_h.copy_(x.to(DEV))
        eager = ops.moe_block(x.to(DEV), gwd, shd, stacked, cfg)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(static_out, eager), f"replay {r}"
        idx, _ = ops.route(x.to(DEV), gwd, cfg)
        routes.add(tuple(idx.flatten().tolist()))
        if r == 0:
            assert_parity(static_out, F.moe_block(x, gw, shared, lambda e: table[e], cfg), "graph replay vs oracle")
    assert len(routes) > 1, "the inputs should route differently"


@pytest.mark.parametrize("d", [256, 384])
def test_moe_experts_groups_at_the_tile_edges(d):
    """Groups around every edge of the row tiles (32, 64, 96 and 128 rows, and more than one tile), a
    hidden size whose last 256-column tile is half, and zero block scales in every projection:
    grouping on the device and on the host against the oracle, and against each other bit for bit
    (a group above 64 rows puts all of them on the tiles, either way)."""
    print(f"[case] moe_experts tile edges d={d}", flush=True)
    rows = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 257]
    E, i, m = len(rows), 256, sum(rows)
    g = torch.Generator().manual_seed(d)
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(m, generator=g)].view(m, 1)
    h = _x((m, d), f"mdev-edge{d}")
    table = {e: _mlp(d, i, f"mdev-edge{e}") for e in range(E)}
    for e in range(E):   # zero scales: first, middle or last K block of one row block
        for k in ("gate_proj", "up_proj", "down_proj"):
            s = table[e][k][1]
            s[e % s.shape[0], e % s.shape[1]] = 0.0
    stacked = _stacked(table, E)
    got, hdr = _run_dev(h, idx, stacked, E, i)
    assert hdr[0] == m and hdr[3] == 0
    assert_parity(got, _want(h, idx, table), f"moe_experts_dev tile edges d={d}")
    tables, _ = ops._stacked_expert_tables(stacked, E, d, torch.device(DEV))
    host = torch.empty(m, 1, d, dtype=torch.bfloat16, device=DEV)
    ops._moe_experts_call(h.to(DEV), idx.contiguous(), tables, i, E, host)
    torch.cuda.synchronize()
    assert torch.equal(host.cpu(), got)


@pytest.mark.parametrize("m,K", [(1, 40), (5, 13), (16, 20)])
def test_moe_experts_dev_few_tokens_repeating_one_expert(m, K):
    """Up to 16 tokens that name one expert over and over: its group is longer than the skinny
    path's rows and is cut into entries of m rows."""
    print(f"[case] moe_experts_dev m={m} K={K} one expert", flush=True)
    E, d, i = 3, 256, 256
    h = _x((m, d), f"mdev-rep{m}")
    idx = torch.ones(m, K, dtype=torch.int64)
    idx[0, 0], idx[m - 1, K - 1] = 0, 2
    table = {e: _mlp(d, i, f"mdev-rep{e}") for e in range(E)}
    got, hdr = _run_dev(h, idx, _stacked(table, E), E, i)
    assert hdr[0] == m * K and hdr[3] == 0
    assert_parity(got, _want(h, idx, table), f"moe_experts_dev repeated m={m} K={K}")


def test_expert_blocks_of_the_smallest_scales():
    """Blocks of zeros under the smallest float scales between ordinary ones (a quantiser that clamps
    their maximum), groups on the tiles of 32 to 128 rows."""
    print("[case] moe_experts smallest scales", flush=True)
    rows, d, i = [20, 40, 70, 110], 384, 384 + 128
    E, m = len(rows), sum(rows)
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows)).view(m, 1)
    h = _x((m, d), "mdev-tiny")
    table = {e: _mlp(d, i, f"mdev-tiny{e}") for e in range(E)}
    for e in range(E):
        for w, s in table[e].values():
            for b in range(s.shape[0]):
                j = (b + e) % s.shape[1]
                z = w[128 * b:128 * b + 128, 128 * j:128 * j + 128]
                z.copy_(torch.zeros_like(z))
                s[b, j] = 2.0 ** -126 if b % 2 else 2.0 ** -149
    stacked = _stacked(table, E)
    got, _ = _run_dev(h, idx, stacked, E, i)
    assert_parity(got, _want(h, idx, table), "smallest scales")


@pytest.mark.parametrize("E,K,m,d,i", [(2, 1, 17, 7168, 2048), (8, 8, 17, 7168, 2048), (8, 8, 32, 7168, 2048),
                                       (4, 2, 33, 7168, 2048), (4, 2, 64, 7168, 2048), (4, 4, 65, 7168, 2048),
                                       (1, 1, 33, 7168, 2048), (24, 2, 33, 7168, 2048), (2, 1, 40, 32896, 256)])
def test_few_experts_on_the_skinny_gemm(E, K, m, d, i):
    """R1's expert shape with few experts, where the tiles would leave most of the machine idle:
    entries of 16 and of 32 rows, groups that end one past them, and the switch at 32 / 33 tokens
    (24 experts: the tiles), on the device and from a host list, against the oracle.  A hidden size
    whose K parts the skinny GEMM cannot add takes the tiles."""
    print(f"[case] moe_experts few experts E={E} K={K} m={m} d={d}", flush=True)
    h = _x((m, d), f"mdev-few{m}-{d}")
    g = torch.Generator().manual_seed(E * 101 + m)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(m)])
    one = [_mlp(d, i, f"mdev-few{d}-{e}") for e in range(min(E, 3))]   # (the weights repeat)
    table = {e: one[e % len(one)] for e in range(E)}
    stacked = _stacked(table, E)
    want = _want(h, idx, table)
    got, hdr = _run_dev(h, idx, stacked, E, i)
    assert hdr[0] == m * K and hdr[3] == 0
    assert_parity(got, want, f"few experts, device E={E} K={K} m={m}")
    tables, _ = ops._stacked_expert_tables(stacked, E, d, torch.device(DEV))
    host = torch.empty(m, K, d, dtype=torch.bfloat16, device=DEV)
    ops._moe_experts_call(h.to(DEV), idx.contiguous(), tables, i, E, host)
    torch.cuda.synchronize()
    assert_parity(host, want, f"few experts, host E={E} K={K} m={m}")


def test_moe_experts_dev_hidden_of_4_gb():
    """Hidden states of more than 4 GB: a gathered row's byte offset does not fit 32 bits.  Rows
    from both ends and the middle equal the same rows in a small call bit for bit (a row's sums do
    not depend on its tile)."""
    m, d, i, E = 65536, 32896, 256, 2
    print(f"[case] moe_experts_dev hidden {m * d * 2 / 2 ** 30:.2f} GiB", flush=True)
    g = torch.Generator(device=DEV).manual_seed(11)
    h = torch.empty(m, d, dtype=torch.bfloat16, device=DEV)
    for r in range(0, m, 8192):
        h[r:r + 8192] = torch.randn(8192, d, generator=g, device=DEV, dtype=torch.bfloat16)
    stacked = {}
    for k, (n, kk) in (("gate_proj", (i, d)), ("up_proj", (i, d)), ("down_proj", (d, i))):
        q = (torch.randn(E, n, kk, generator=g, device=DEV) * 60).clamp(-448, 448).to(torch.float8_e4m3fn)
        stacked[k] = (q, torch.rand(E, n // 128, kk // 128, generator=g, device=DEV) * 1e-3)
    idx = torch.arange(m, device=DEV).remainder(3).clamp(max=1).view(m, 1)
    table, n_inter = ops._stacked_device_table(stacked, E, d, torch.device(DEV))
    out = torch.empty(m, 1, d, dtype=torch.bfloat16, device=DEV)
    ops._moe_experts_dev_call(h, idx, table, n_inter, E, out)
    # (more than 64 rows per expert: on the tiles, as in the large call)
    rows = torch.cat([torch.arange(0, 100), torch.arange(32700, 32800), torch.arange(m - 100, m)]).to(DEV)
    few = torch.empty(rows.numel(), 1, d, dtype=torch.bfloat16, device=DEV)
    ops._moe_experts_dev_call(h[rows].contiguous(), idx[rows].contiguous(), table, n_inter, E, few)
    torch.cuda.synchronize()
    assert torch.isfinite(few.float()).all() and few.float().abs().max() > 0
    assert torch.equal(out[rows], few)
