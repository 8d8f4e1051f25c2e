"""What amla_mla_prefill_workspace_bytes says of a prefill of R1's layer: its fixed rows and K-part
sums by the sizes of the layer, and so the attention's own scratch, which tells its form."""
import ctypes

from amla._lib import MlaArgs, lib

LINEARS = ((1536 + 576, 7168), (128 * 192, 1536), (7168, 128 * 128))   # q_a | kv_a, q_b, o_proj


def _up(nbytes):
    return -(-nbytes // 256) * 256


def size(batch, new, rows):
    a = MlaArgs()
    a.batch, a.seq_len, a.hidden, a.heads, a.q_lora, a.kv_lora = batch, new, 7168, 128, 1536, 512
    a.qk_nope, a.qk_rope, a.v_dim, a.max_seq, a.rope_rows, a.max_context = 128, 64, 128, rows, rows, rows
    return lib().amla_mla_prefill_workspace_bytes(ctypes.byref(a))


def _fixed_and_sums(batch, new):
    """Normed and projected rows; K-part sums of the linears at this and, below it, at the smaller
    row counts where the skinny linears' plans change."""
    m = batch * new
    fixed = sum(_up(m * c * 2) for c in (7168, 1536, 1536, 128 * 192, 128 * 128))
    at = [m, *[t for t in (8, 16, 32, 64) if t < m]]
    return fixed, max(lib().amla_fp8_linear_workspace_bytes(t, n, k) for n, k in LINEARS for t in at)


def scratch(batch, new, rows):
    """Bytes of a latent attention's scratch."""
    fixed, sums = _fixed_and_sums(batch, new)
    return size(batch, new, rows) - fixed - _up(sums)


def runs_latent(batch, new, rows):
    """The decompressed form holds normed rows, rope keys and kv_b rows of one sequence."""
    fixed, sums = _fixed_and_sums(batch, new)
    sums = max(sums, lib().amla_fp8_linear_workspace_bytes(rows, 128 * 256, 512))
    return size(batch, new, rows) != fixed + _up(rows * 512 * 2) + _up(rows * 64 * 2) + _up(rows * 128 * 256 * 2) + _up(sums)
