"""A prompt chunk's layers: many consecutive token rows at once (hsd/model.py:259-279 runs a
prompt in chunks through the blocks).

`prep` normalises the rows once per projection (the bits of nn.linear's prologue), `gemm`
multiplies them with a 4-bit or bf16 weight, and `moe_up` runs every expert's up projection
with ReLU^2 over the (token, slot) pairs sorted by expert. The arithmetic is nn.linear's and
moe.up_relu2's with the matrix cores' summation order. `scan` and `attention` are the
Mamba-2 recurrence and the causal attention of the chunk's rows at positions *pos .. of a
prompt of `total` tokens.
"""
from __future__ import annotations

import ctypes
import math

import torch

from . import _native as N
from .prefill import num_tiles


def group_pitch(I):
    """Group sums per row and part: I/64 rounded up to 8."""
    return (I // 64 + 7) // 8 * 8


def moe_rows(D, F, FS, topk):
    """The most rows of one moe_up or moe_down call: each of its buffers (h, the group sums, the
    slots' partial sums) stays below 1 GiB."""
    row = max(2 * (topk * F + FS), 6 * (topk + 1) * group_pitch(max(F, FS)), 4 * (topk + 1) * D)
    return max(((1 << 30) - 1) // row, 1)


class Rows:
    """Prepared rows: xp [T, I] bf16 and, for 4-bit weights, the group sums hs [T, 3 GP]."""

    def __init__(self, xp, hs):
        self.xp, self.hs = xp, hs


def prep(x, norm=None, eps=1e-5, gated_z=False, sums=True):
    """x [T, I]: bf16 rows (norm: the RMS norm's weight), or with gated_z mamba's z rows (f32,
    I + I/16 values per row) and the gated norm's weight. sums: for 4-bit weights."""
    T, I = x.shape
    ld, unit = x.stride()
    if unit != 1 or x.dtype != (torch.float32 if gated_z else torch.bfloat16):
        raise N.HSDError("prep takes unit-stride bf16 rows, or gated_z's f32 rows")
    if gated_z and norm is None:
        raise N.HSDError("gated_z takes a norm weight")
    kind = N.X_GATED_Z if gated_z else N.X_RMS if norm is not None else N.X_BF16
    xp = torch.empty((T, I), dtype=torch.bfloat16, device=x.device)
    hs = torch.empty((T, 3 * group_pitch(I)), dtype=torch.bfloat16, device=x.device) if sums else None
    N.call("hsd_rows_prep", x, ld, kind, norm, float(eps), xp, hs, T, I,
           N.stream(x.device))
    return Rows(xp, hs)


def _row_stride(t, T, O):
    ld, unit = t.stride()
    if t.dtype != torch.bfloat16 or unit != 1 or t.shape != (T, O):
        raise N.HSDError(f"gemm: out and residual must be unit-stride bf16 rows [{T}, {O}]")
    return ld


def gemm(rows: Rows, W, residual=None, out=None):
    """bf16 y [T, O] = xn W^T (W: nn.QWeight); residual: y = bf16(residual + bf16(xn W^T))
    (4-bit weights; out may be residual)."""
    xp, hs = rows.xp, rows.hs
    T, I = xp.shape
    q4, y, rld = W.q4, out, 0
    if I != W.I:
        raise N.HSDError(f"gemm: the rows have {I} inputs, the weight {W.I}")
    if q4 and hs is None:
        raise N.HSDError("gemm: a 4-bit weight takes rows prepared with their group sums")
    if residual is not None:
        if not q4:
            raise N.HSDError("gemm: a residual is added to a 4-bit weight's product only")
        rld = _row_stride(residual, T, W.O)
    if out is None:
        y, ld = torch.empty((T, W.O), dtype=torch.bfloat16, device=xp.device), W.O
    else:
        ld = rld if out is residual else _row_stride(out, T, W.O)
    st = N.stream(xp.device)
    if q4:
        N.call("hsd_gemm_q4", xp, hs, W.w, W.scales, W.biases, y, ld, residual, rld, T, W.O, I, st)
    else:
        N.call("hsd_gemm_bf16", xp, I, 0 if hs is None else 1, W.w, y, ld, T, W.O, I, st)
    return y


def moe_tiles(sel, E, tt, status=None):
    """prefill.build_tiles' lists and the routed tiles in use: (tile_e, tile_slot, ntiles [1])."""
    T, K = sel.shape
    NT = num_tiles(T, K, E, tt)
    t = torch.empty(NT * (tt + 1) + 1, dtype=torch.int32, device=sel.device)
    tile_e, tile_slot, ntiles = t[:NT], t[NT:NT * (tt + 1)], t[NT * (tt + 1):]
    N.call("hsd_moe_tiles", sel, T, K, E, tt, tile_e, tile_slot, ntiles, status,
           N.stream(sel.device))
    return tile_e, tile_slot, ntiles


def moe_up(rows: Rows, tiles, w1, s1, b1, sw1, ss1, sb1, *, topk, tt):
    """moe.up_relu2 of a chunk -> (hcat [T, topk*F + FS] bf16, its 64-neuron group sums)."""
    T, D = rows.xp.shape
    E, F, FS = w1.shape[0], w1.shape[1], sw1.shape[0]
    hcat = torch.empty((T, topk * F + FS), dtype=torch.bfloat16, device=rows.xp.device)
    hsum = torch.empty((T, topk + 1, 3 * group_pitch(max(F, FS))), dtype=torch.bfloat16, device=rows.xp.device)
    N.call("hsd_moe_up_gemm", rows.xp, rows.hs, tiles[0], tiles[1], tiles[2],
           N.as_words(N.contig(w1)), N.contig(s1), N.contig(b1), N.as_words(N.contig(sw1)), N.contig(ss1),
           N.contig(sb1), hcat, hsum, T, D, F, FS, topk, E, tt, N.stream(rows.xp.device))
    return hcat, hsum


def moe_down(x, hcat, hsum, sel, gains, tiles, pw, ps, pb, spw, sps, spb, *, topk, tt, out=None):
    """bf16(x + bf16(the MoE down projection)) of a chunk, every row of the neuron-major layout
    read (out may be x)."""
    T, D = x.shape
    E, F, FS = pw.shape[0], pw.shape[1], spw.shape[0]
    y = out if out is not None else torch.empty((T, D), dtype=torch.bfloat16, device=x.device)
    nb = N.call("hsd_moe_down_workspace_bytes", T, D, topk)
    ws = torch.empty(nb, dtype=torch.uint8, device=x.device)
    N.call("hsd_moe_down_gemm", hcat, hsum, sel, gains, tiles[0], tiles[1],
           tiles[2], N.as_words(N.contig(pw)), N.contig(ps), N.contig(pb), N.as_words(N.contig(spw)), N.contig(sps),
           N.contig(spb),
           x, x.stride(0), y, y.stride(0), T, D, F, FS, topk, E, tt, ws, nb, N.stream(x.device))
    return y


def scan(mixer, proj, cache, pos, total, status=None):
    """mamba.ssm_rows(..., gated=True) of a chunk from the in_proj output [T, 2*H*P + 2*G*N + H]:
    -> z [T, H*P] f32 (a view of rows of H*P + H*P/16 values); the state after the chunk goes to
    the ring slab the advanced ring index names."""
    T = proj.shape[0]
    H, P, Nst, G = mixer.num_heads, mixer.head_dim, mixer.ssm_state_size, mixer.n_groups
    DI, CD = mixer.intermediate_size, mixer.conv_dim
    ld, unit = proj.stride()
    if unit != 1 or proj.dtype != torch.bfloat16 or proj.shape[1] < DI + CD + H:
        raise N.HSDError(f"proj needs {DI + CD + H} unit-stride bf16 columns")
    z = torch.empty((T, DI + DI // 16), dtype=torch.float32, device=proj.device)
    nb = N.call("hsd_mamba_scan_workspace_bytes", T, H, P, Nst, G)
    ws = torch.empty(nb, dtype=torch.uint8, device=proj.device)
    base, es = proj.data_ptr(), 2
    lo, hi = mixer.time_step_limit
    N.call("hsd_mamba_scan", ctypes.c_void_p(base + DI * es), ld, ctypes.c_void_p(base + (DI + CD) * es), ld, proj,
           ld, N.contig(mixer.conv_w), N.contig(mixer.conv_b), N.contig(mixer.A_log),
           N.contig(mixer.dt_bias), N.contig(mixer.D), cache.ssm, cache.conv,
           cache.cur, cache.nslab, pos, z, z.stride(0), T, total, H, P, Nst, G, float(lo), float(hi),
           status, ws, nb, N.stream(proj.device))
    return z[:, :DI]


def attention(qkv, kv, pos, total, *, n_heads, n_kv_heads, head_dim=128, status=None):
    """nn.attention of a chunk: the rows' keys and values into the cache, then causal attention
    -> [T, HQ*HD] bf16."""
    T = qkv.shape[0]
    out = torch.empty((T, n_heads * head_dim), dtype=torch.bfloat16, device=qkv.device)
    N.call("hsd_attn_prompt", qkv, qkv.stride(0), T, total, kv.k, kv.v, kv.smax, pos,
           out, out.stride(0), n_heads, n_kv_heads, head_dim, 1.0 / math.sqrt(head_dim),
           status, N.stream(qkv.device))
    return out


def kv_append(kvrows, kv, pos, total, *, n_kv_heads, head_dim=128, status=None):
    """The keys and values of a chunk's rows (kvrows [T, 2*HKV*HD]: k | v) into the cache."""
    N.call("hsd_kv_append", kvrows, kvrows.stride(0), kvrows.shape[0], total, kv.k, kv.v, kv.smax, pos, n_kv_heads,
           head_dim, status, N.stream(kvrows.device))
