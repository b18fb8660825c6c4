"""Causal prefill attention of the full-attention layers: stands where the reference calls
mx.fast.scaled_dot_product_attention(q, K[:, :, :kv_len], V[:, :, :kv_len], scale=D**-0.5, mask="causal")
(qwen35/model.py:160-167, qwen35/prefill.py:468).  8 query heads on 2 KV heads, head dim 256."""
from __future__ import annotations

from . import _lib as L


def scaled_dot_product_attention(q, k, v, *, scale: float, mask="causal"):
    """q [1, 8, S, 256], k / v [1, 2, L, 256] bf16 (k, v may be length-slices of a longer cache).  mask = "causal": query i
    sits at position L - S + i and sees keys 0 .. L - S + i.  Returns [1, 8, S, 256] bf16 in q's memory layout: head-major, or
    token-major if q is the transposed view of [S, 8, 256] rows (what qkv_prep returns and out_gate takes); neither is copied."""
    if mask != "causal":
        raise ValueError("only mask='causal' is built (decode / verify rows go through batch.attn_b)")
    if abs(scale - 256 ** -0.5) > 1e-9:
        raise ValueError("only scale = 256**-0.5 is built")
    return L.host.sdpa(q, k, v)


QKV_W = 8 * 512 + 2 * 2 * 256


def qkv_prep(qkv, q_norm, k_norm, pos, M=1, eps=1e-6, max_pos=None):
    """The steps between the qkv projection and the attention kernel of a full-attention layer (qwen35/batch.py:505-512,
    qwen35/model.py:154-164): split the 5120-wide rows into q / gate / k / v, RMS-normalise q and k per head (weights [256]
    bf16), rotate their first 64 features to the row's position.  qkv [R,5120] bf16, pos int32 [R / M] (row b*M + j sits at
    pos[b] + j).  Returns q [R,8,256], k [R,2,256], v [R,2,256] bf16; the gate stays in qkv (out_gate reads it there).
    max_pos: a bound of the positions that the caller knows on the host (a prefill knows its key count): the rotary (cos,
    sin) pairs then come from the device's table of positions 0 .. max_pos instead of being evaluated per row (same bits;
    a row beyond the bound still evaluates its own)."""
    return L.host.qkv_prep(qkv, q_norm, k_norm, pos, M, eps, max_pos)


def out_gate(o, qkv):
    """o * sigmoid(gate) (qwen35/batch.py:513): o [R,8,256] bf16, qkv [R,5120] bf16 -> [R,2048] bf16"""
    return L.host.out_gate(o, qkv)
