"""The GEMM tiles of fp8_linear / swiglu above 64 rows at their edges: row counts around the 32-row
steps and the 128-row tiles, output columns that end inside a tile, a 128-row segment or a scale
block, K from one block up, zero block scales, K parts or none, row strides without 16-byte
alignment, fp32 rows.

The reference is a float64 product of the same operands.  fp32 sums of at most 2304 products of
magnitude about |x| |w| stay within 2e-5 of the row's norm (eps32 * sqrt(K) and the scale ratios'
K / 128 roundings, with a factor of 4); bf16 outputs add half a bf16 ulp (2^-9)."""
import pytest
import torch

from amla import ops, synth
from amla._lib import lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(m, n, k, tag, zero=()):
    w, s = synth.quantize_fp8_blocks(synth.randn((n, k), synth.seed_of("tile", tag, n, k), 0.05))
    for i, j in zero:
        s[i % s.shape[0], j % s.shape[1]] = 0.0
    x = synth.randn((m, k), synth.seed_of("tile-x", tag, m, k), 1.0).to(torch.bfloat16)
    full = w.double() * s.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    want = x.double() @ full.T
    bound = 2e-5 * (x.double().norm(dim=1)[:, None] * full.norm(dim=1)[None, :]) + 1e-30
    return x.to(DEV), w.to(DEV), s.to(DEV), want, bound


def _check(got, want, bound, bf16):
    d = (got.double().cpu() - want).abs()
    lim = bound + (want.abs() * 2.0 ** -8 if bf16 else 0)
    assert torch.isfinite(got.float()).all()
    assert bool((d <= lim).all()), f"max excess {(d - lim).max().item():.3e}"


def _raw(x, w, s, ldy, f32, ws):
    """amla_fp8_linear(_f32) with an output row stride and a workspace of `ws` bytes (None: NULL)."""
    m, k = x.shape
    n = w.shape[0]
    y = torch.full((m, ldy), -7.0, dtype=torch.float32 if f32 else torch.bfloat16, device=DEV)
    buf = torch.empty(ws, dtype=torch.uint8, device=DEV) if ws else None
    fn = lib().amla_fp8_linear_f32 if f32 else lib().amla_fp8_linear
    ops.check(fn(x.data_ptr(), m, k, k, w.data_ptr(), s.data_ptr(), n, y.data_ptr(), ldy,
                 buf.data_ptr() if buf is not None else None, ws or 0, ops._stream_ptr(x)), "fp8_linear")
    assert (y[:, n:] == -7.0).all(), "columns past n were written"
    return y[:, :n]


@pytest.mark.parametrize("m,n,k", [(65, 128, 128), (96, 144, 256), (97, 256, 384), (128, 272, 640), (129, 384, 128),
                                   (160, 576, 2304), (191, 16, 1152), (257, 1040, 512), (300, 784, 1536)])
@pytest.mark.parametrize("f32", [False, True])
def test_tiles_and_k_parts(m, n, k, f32):
    print(f"[case] tile linear m={m} n={n} k={k} f32={f32}", flush=True)
    x, w, s, want, bound = _case(m, n, k, "edge", zero=((0, 0), (1, 1), (2, k // 128 - 1)))
    need = lib().amla_fp8_linear_workspace_bytes(m, n, k)
    assert k < 1152 or need > 0, "a few tiles of a long K should be cut into parts"
    for ws in {need or None, None}:
        _check(_raw(x, w, s, n, f32, ws), want, bound, not f32)
        _check(_raw(x, w, s, n + 4, f32, ws), want, bound, not f32)     # 8-byte aligned bf16 rows
    got = ops.fp8_linear(x, w, s, torch.float32 if f32 else torch.bfloat16)
    _check(got, want, bound, not f32)


@pytest.mark.parametrize("m,n,k", [(128 * 65, 256 * 8, 1152), (384, 256 * 173, 1152), (896, 256 * 74, 1152)])
def test_many_tiles_end_in_parts(m, n, k):
    """More tiles than one round of the machine (512): whole tiles first, the rest in K parts; 65 row
    tiles, and 3 and 7 of them, which do not divide the round (a column tile's row tiles are then
    split between the two)."""
    tiles, need = -(-m // 128) * (n // 256), lib().amla_fp8_linear_workspace_bytes(m, n, k)
    print(f"[case] tile linear {tiles} tiles, workspace {need}", flush=True)
    rest, part = tiles - 512, 256 * 128 * 4
    assert 0 < rest < 64 and need % (rest * part) == 0 and 2 <= need // (rest * part) <= 16
    x, w, s, want, bound = _case(m, n, k, "many")
    _check(ops.fp8_linear(x, w, s), want, bound, True)


@pytest.mark.parametrize("m,n,k", [(130, 256 * 130, 2304), (1200, 256 * 27, 2304)])
def test_one_tile_per_cu_and_parts_beside_it(m, n, k):
    """A little more than 256 tiles: 256 (or the row tiles of as many whole column tiles) run whole,
    the rest in K parts beside them."""
    print(f"[case] tile linear m={m} n={n} k={k}", flush=True)
    x, w, s, want, bound = _case(m, n, k, "beside")
    assert lib().amla_fp8_linear_workspace_bytes(m, n, k) > 0
    _check(ops.fp8_linear(x, w, s), want, bound, True)


@pytest.mark.parametrize("m,n,k", [(65, 128, 256), (100, 384, 1152), (129, 256, 128), (333, 640, 768)])
def test_swiglu_tiles(m, n, k):
    """silu(gate) * up in the tile's epilogue and in the K-part finish, intermediate sizes that are
    an odd multiple of 128, a zero scale in each weight; against float64 with the bf16 roundings of
    the reference (gate, up, silu, product)."""
    print(f"[case] swiglu tiles m={m} n={n} k={k}", flush=True)
    x, gw, gs, g, _ = _case(m, n, k, "gate", zero=((0, 1),))
    _, uw, us, _, _ = _case(m, n, k, "up", zero=((1, 0),))
    full = uw.double().cpu() * us.double().cpu().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    u = x.double().cpu() @ full.T
    dw, ds = synth.quantize_fp8_blocks(synth.randn((k, n), synth.seed_of("tile-down", n, k), 0.05))
    r = lambda t: t.to(torch.bfloat16).double()
    g, u = r(g), r(u)
    h = r(r(g / (1.0 + torch.exp(-g))) * u)
    dfull = dw.double() * ds.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    want = h @ dfull.T
    got = ops.swiglu(x, gw, gs, uw, us, dw.to(DEV), ds.to(DEV)).double().cpu()
    # an fp32 sum next to a rounding boundary may move g or u by one bf16 ulp: h then differs by 2^-7 in few entries
    # (one K block of zero scales in either weight makes the whole output zero at k = 128: it must be so)
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("m,stride", [(130, 4096 * 7168), (192, 36000000)])
@pytest.mark.parametrize("f32", [False, True])
def test_rows_four_gb_apart(m, stride, f32):
    """x rows so far apart that a row's byte offset in its tile does not fit 32 bits (130 rows: the
    last positions of sequences of 4096 tokens; 192: in the tile of 64 rows too): the same bits as
    packed rows."""
    k, n = 640, 272
    print(f"[case] tile linear m={m} row stride {stride}", flush=True)
    x, w, s, want, bound = _case(m, n, k, "far")
    far = torch.empty(m, stride, dtype=torch.bfloat16, device=DEV)[:, :k]
    far.copy_(x)
    out = torch.float32 if f32 else torch.bfloat16
    got = ops.fp8_linear(far, w, s, out)
    assert torch.equal(got, ops.fp8_linear(x, w, s, out))
    _check(got, want, bound, not f32)


@pytest.mark.parametrize("m,n,k", [(100, 384, 640), (129, 256, 1152), (160, 144, 2304)])
def test_blocks_of_the_smallest_scales(m, n, k):
    """Blocks of zeros under the smallest normal and denormal scales (a quantiser that clamps their
    maximum) between ordinary blocks, and small values under a scale of 2^-80: in 96 and 128-row
    tiles and in those of whole lines, with K parts and without."""
    print(f"[case] tile linear smallest scales m={m} n={n} k={k}", flush=True)
    x, w, s, _, _ = _case(m, n, k, "tiny")
    w, s, nb, kb = w.cpu(), s.cpu(), -(-n // 128), k // 128
    blk = lambda i, j: (slice(128 * i, 128 * i + 128), slice(128 * j, 128 * j + 128))
    for i in range(nb):
        for j, v in (((i + 1) % kb, 2.0 ** -126), ((i + 3) % kb, 2.0 ** -149)):
            w[blk(i, j)] = torch.zeros_like(w[blk(i, j)])
            s[i, j] = v
    s[nb - 1, kb - 1] = 2.0 ** -80
    full = w.double() * s.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    want = x.double().cpu() @ full.T
    bound = 2e-5 * (x.double().cpu().norm(dim=1)[:, None] * full.norm(dim=1)[None, :]) + 1e-30
    need = lib().amla_fp8_linear_workspace_bytes(m, n, k)
    wd, sd = w.to(DEV), s.to(DEV)
    for ws in {need or None, None}:
        _check(_raw(x, wd, sd, n, False, ws), want, bound, True)
        _check(_raw(x, wd, sd, n, True, ws), want, bound, False)
