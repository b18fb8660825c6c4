"""Batched decode for B independent sequences at different positions: the call surface of qwen35/batch.py.

State lives in slot pools that the kernels update in place (qwen35/batch.py:1-18):
  ssm  : [S+1, 16, 128, 128] float32      slot s = one sequence
  conv : [(S+1)*2, 3, 6144]  bf16          double buffered: a step reads buffer pos&1 and writes the other one
  K, V : [S+1, 2, Lmax, 256] bf16          the attention kernel appends the new row of each sequence at its position
  slot S is the trash slot that padding rows point at.
All launches go to the current torch stream; in-place writes are ordered by stream order."""
from __future__ import annotations

import torch

from . import _lib as L
from .model import Cfg

BF16 = torch.bfloat16
HV, DK, DV, CD, PW = 16, 128, 128, 6144, 8224


def deltanet_b(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, rows_per_wg: int = 0):
    """proj [B, 8224] bf16; slots / pos int32 [B] (pos = tokens already in the slot's state).  Returns y [B, 2048] bf16 and
    updates ssm_pool[slot] and the conv buffer (pos&1)^1 of the slot IN PLACE (qwen35/batch.py:128-135)."""
    return L.host.decode_step(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, rows_per_wg)


def deltanet_b_gnorm(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, gw, eps=1e-6):
    """deltanet_b followed by gnorm_rows (qwen35/batch.py:128-135, 338-343; the two calls of the reference's decode step,
    batch.py:497-499) in one launch.  Returns the gated-norm output [B, 2048] bf16 (the same bits as the two calls); pools are
    updated in place as by deltanet_b."""
    return L.host.decode_step_gnorm(proj, conv_pool, conv_w, A_log, dt_bias, ssm_pool, slots, pos, gw, eps)


def split_size(Lmax: int, B: int = 16) -> int:
    """Smallest number of pool keys a split-K workgroup takes.  The kernel spreads the batch's key tiles evenly over one
    workgroup per CU whatever the mix of lengths; this lower bound only matters for small batches of short sequences (layer form, us,
    with 32 / 64 / 128 keys: 5 x 3 of 90 - 900 12.4 / 12.5 / 14.6, 16 of 100 - 1000 13.7 / 13.7 / 15.0, one sequence of 300 9.3 / 9.6 / 10.3, of 1000
    9.7 / 9.7 / 10.8, of 2000 10.9 / 10.2 / 13.4, of 4000 12.8 / 12.1 / 11.8, of 8000 13.6 / 13.5 / 14.3, of 16000 16.1 / 15.9 / 15.7, and with four rows 11.0 /
    11.1 / 11.4, 11.4 / 11.2 / 12.3, 12.8 / 11.6 / 15.5, 15.1 / 14.1 / 13.2, 15.7 / 15.6 / 16.7, 18.3 / 18.2 / 18.1)."""
    return 32


def attn_b(q, k, v, Kp, Vp, slots, pos, M=1, split=None, workspace=None):
    """q [R,H,D], k / v [R,KV,D] (normed + roped), pools [S+1,KV,Lmax,D]; R = B*M rows (row b*M+j = position pos[b]+j of slot
    slots[b]; slots / pos int32 [B]).  Returns o [R,H,D] bf16 and appends k / v at pos[b]+j (in place)
    (qwen35/batch.py:230-237).  M up to 16 (the limit of batch_spec.deltanet_bm); more than four tokens per sequence run as
    passes of four, each reading the pool once.  workspace: optional uint8 device tensor of at least qt_gqa_attn_workspace_bytes(B, M, Lmax, split)
    bytes for the split-K partial results (default: a buffer cached per device and stream; under HIP graph capture, memory of the graph)."""
    return L.host.attn_b(q, k, v, Kp, Vp, slots, pos, M, split or split_size(0), workspace)


def attn_layer_b(qkv, q_norm, k_norm, Kp, Vp, slots, pos, M=1, eps=1e-6, split=None, workspace=None):
    """The attention half of a full-attention layer at a decode / verify step (qwen35/batch.py:505-513), between the qkv and o
    projections: q / k RMSNorm and rotary embedding, attn_b, and o * sigmoid(gate), in two launches per pass of four tokens
    (attention.qkv_prep + attn_b + attention.out_gate are four), with the same bits.  qkv [B*M,5120] bf16 = [(q_h | gate_h) x 8 |
    k x 2 | v x 2]; q_norm, k_norm [256] bf16; pools, slots, pos, M as for attn_b (the new K / V rows are appended in place).
    Returns [B*M,2048] bf16.  The first call on a device (and the first one with a longer pool) builds the rotary table and
    waits for it; under HIP graph capture the table belongs to the graph, and every replay of such a call writes it again."""
    return L.host.attn_layer_b(qkv, q_norm, k_norm, Kp, Vp, slots, pos, M, eps, split or split_size(0), workspace)


def gnorm_rows(y, proj, gw, eps=1e-6):
    """Gated RMSNorm of the delta-rule output (qwen35/batch.py:338-343): y [B, 2048] bf16, proj [B, 8224] bf16 (its z slice
    is at 6144:8192), gw float32 [128].  Returns [B, 2048] bf16."""
    return L.host.gated_norm(y, proj, gw, eps)


def rms_rows(x, nw, eps=1e-6, T=128, f32=False):
    """qwen35/batch.py:295-301; see kernels.rms_rows."""
    from .kernels import rms_rows as _rms_rows
    return _rms_rows(x, nw, eps, T, f32)


def blit(dst, src, n, d0, s0, ny=1, dstride=0, sstride=0):
    """dst.flat[d0 + y*dstride + i] = src.flat[s0 + y*sstride + i] for i < n, y < ny, in place (qwen35/batch.py:365-372).
    dst and src are contiguous device tensors of the same dtype (bf16 or float32); returns dst."""
    if dst.dtype != src.dtype or dst.dtype not in (BF16, torch.float32):
        raise TypeError(f"blit: bf16 or float32 tensors of one dtype expected, got {dst.dtype} and {src.dtype}")
    dst, src = L.dev(dst, dst.dtype, "dst"), L.dev(src, src.dtype, "src")
    n, d0, s0, ny, dstride, sstride = (int(x) for x in (n, d0, s0, ny, dstride, sstride))
    if n < 0 or ny < 0 or min(d0, s0, dstride, sstride) < 0:
        raise ValueError("blit: negative size, offset or stride")
    if n and ny and (d0 + (ny - 1) * dstride + n > dst.numel() or s0 + (ny - 1) * sstride + n > src.numel()):
        raise ValueError("blit: the copy leaves the source or the destination")
    L.call("qt_blit", L.ptr(dst), L.ptr(src), dst.element_size(), n, d0, s0, ny, dstride, sstride, L.stream())
    return dst


def blit_batch(jobs):
    """Several blits in one launch: jobs = [(dst, src, n, d0, s0, ny, dstride, sstride), ...] with the arguments of blit.
    Every copy must be 16-byte granular (a ValueError says which one is not)."""
    L.host.blit_batch(jobs, ())


class Pools:
    """Slot-major state pools of the batched decode step (qwen35/batch.py:405-462)."""

    def __init__(self, cfg: Cfg, slots: int, max_len: int, device="cuda"):
        self.cfg, self.S, self.Lmax = cfg, slots, max_len
        nl = sum(cfg.is_linear(i) for i in range(cfg.layers))
        na = cfg.layers - nl
        z = lambda shape, dt: torch.zeros(shape, dtype=dt, device=device)
        self.conv = [z(((slots + 1) * 2, 3, CD), BF16) for _ in range(nl)]
        self.ssm = [z((slots + 1, HV, DV, DK), torch.float32) for _ in range(nl)]
        self.K = [z((slots + 1, cfg.n_kv, max_len, cfg.head_dim), BF16) for _ in range(na)]
        self.V = [z((slots + 1, cfg.n_kv, max_len, cfg.head_dim), BF16) for _ in range(na)]

    def nbytes(self):
        return sum(a.numel() * a.element_size() for g in (self.conv, self.ssm, self.K, self.V) for a in g)

    @staticmethod
    def slot_bytes(cfg: Cfg, max_len: int, double_conv=True):
        """Bytes one sequence occupies in the pools (qwen35/batch.py:420-426)."""
        nl = sum(cfg.is_linear(i) for i in range(cfg.layers))
        na = cfg.layers - nl
        return (nl * (HV * DV * DK * 4 + (2 if double_conv else 1) * 3 * CD * 2)
                + na * 2 * cfg.n_kv * max_len * cfg.head_dim * 2)

    def as_tree(self):
        return {"conv": self.conv, "ssm": self.ssm, "K": self.K, "V": self.V}

    def load(self, slot: int, state: dict, pos: int):
        """Copy a prefilled single-sequence state (kv [1,2,max_len,256] pairs, conv [1,3,6144], ssm [1,16,128,128], valid after
        `pos` tokens) into `slot`, in place, with the strided copy kernel (qwen35/batch.py:431-447)."""
        assert 0 <= slot < self.S and 0 < pos <= self.Lmax, (slot, pos)
        L.host.pools_load(self.conv, self.ssm, self.K, self.V, state["conv"], state["ssm"], state["kv"], slot, pos, self.Lmax,
                          self.cfg.n_kv, self.cfg.head_dim)      # one launch for the whole sequence (the reference issues 48 blits)

    def read(self, slot: int, pos: int, max_len: int | None = None):
        """The slot's state as a single-sequence state dict of fresh tensors (qwen35/batch.py:449-462): the inverse of load,
        one launch of the strided copy kernel; K / V rows from `pos` on are zero."""
        ml = max_len or self.Lmax
        par = pos & 1
        nkv, D = self.cfg.n_kv, self.cfg.head_dim
        n = min(pos, ml)
        st = {"kv": [], "conv": [torch.empty((1, 3, CD), dtype=BF16, device=c.device) for c in self.conv],
              "ssm": [torch.empty((1, HV, DV, DK), dtype=torch.float32, device=s.device) for s in self.ssm]}
        jobs = []
        for i in range(len(self.conv)):
            jobs.append((st["conv"][i], self.conv[i], 3 * CD, 0, (slot * 2 + par) * 3 * CD, 1, 0, 0))
            jobs.append((st["ssm"][i], self.ssm[i], HV * DV * DK, 0, slot * HV * DV * DK, 1, 0, 0))
        for K, V in zip(self.K, self.V):
            pair = []
            for P in (K, V):
                out = torch.zeros((1, nkv, ml, D), dtype=P.dtype, device=P.device)
                if n:
                    jobs.append((out, P, n * D, 0, slot * nkv * self.Lmax * D, nkv, ml * D, self.Lmax * D))
                pair.append(out)
            st["kv"].append(tuple(pair))
        blit_batch(jobs)
        return st
