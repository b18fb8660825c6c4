"""Two-phase chunked gated-delta-rule for prefill: the call surface of qwen35/gdn_nax.py (prep_a, phase_b, gdn_chunked).

Chunk size is 64 (the reference's is 16; the chunked form is an identity for every chunk size).  The three buffers that
travel from phase A to phase B keep the reference's argument slots (Tbuf, Abuf, gv) but hold this implementation's own
records: the packed half-precision MFMA operands, the U tiles (half precision), and the per-token / per-chunk decay factors."""
from __future__ import annotations

import torch

from . import _lib as L

BF16 = torch.bfloat16
HV, DK, DV, CD, PW = 16, 128, 128, 6144, 8224
CHUNK = 64

# precision flags of the reference (qwen35/gdn_nax.py:363-366) are accepted and ignored: the operands are always fp16
FLAGS = ("RNE", "SPLIT_P1", "SPLIT_P2", "SPLIT_D", "SPLIT_Y", "SPLIT_DP", "PF")
DEFAULT_FLAGS = frozenset()
TG = 64


def _phase_a(proj, conv_state, conv_w, A_log, dt_bias, qkv=None, want_qkv=True, conv_out=None):
    """Phase A.  With q, k, v given: the kernel that consumes them.  Otherwise one kernel that convolves and normalizes the
    projection rows itself (returning q, k, v only if want_qkv) and, if conv_out [3,6144] is given, writes the new conv
    window there.  Returns (q, k, v, ops, U, gC)."""
    return L.host.phase_a(proj, conv_state, conv_w, A_log, dt_bias, qkv, want_qkv, conv_out)


def prep_a(proj, conv_state, conv_w, A_log, dt_bias, relaxed=True):
    """conv+silu+qk-norm and phase A in one launch (qwen35/gdn_nax.py:394-401).
    proj [S,8224], conv_state [3,6144], conv_w [6144,4,1] -> q, k, v [S,16,128] bf16 and the three phase-B records."""
    return _phase_a(proj, conv_state, conv_w, A_log, dt_bias)


def gdn_chunked(q, k, v, proj, A_log, dt_bias, state, relaxed=True, flags=DEFAULT_FLAGS, tg=None):
    """q,k,v [S,16,128] bf16 (q/k already normalized + scaled), proj [S,8224] bf16 (b at 8192:8208, a at 8208:8224),
    state [1,16,128,128] fp32.  Returns y [S,16,128] bf16, new_state [1,16,128,128] fp32  (qwen35/gdn_nax.py:413-426)."""
    _, _, _, ops, U, gC = _phase_a(proj, None, None, A_log, dt_bias, qkv=(q, k, v))
    return phase_b(q, k, v, ops, U, gC, state)


_SNAP = {}            # (device index, stream handle) -> float16 tensor: flag area + chain snapshots
_SNAP_RETIRED = []    # outgrown buffers stay alive: a captured HIP graph may hold their address
_STATUS = {}          # (device index, stream handle) -> pinned int32[2]: set to 1 by a launch that gave up / whose values are not finite

GAVE_UP, NOT_FINITE = 1, 2        # bits of the status word


class ChunkedPrefillError(RuntimeError):
    """A chunked-prefill launch on this stream reported a failure in its status word: its results are not to be used."""


def _key(dev):
    return (dev.index if dev.index is not None else torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)


def _snap_buffer(dev, nbytes):
    """The buffer between phase B's chain and output workgroups, cached per (device, stream): its first 33 KiB are the flag
    area, which has to be zero before a launch and is left zero by it, so the buffer is zero-filled once, when it is made."""
    key = _key(dev)
    buf = _SNAP.get(key)
    if buf is None or buf.numel() * 2 < nbytes:
        if buf is not None:
            torch.cuda.current_stream(dev).synchronize()
            _raise_if_failed([key])                        # what the launches with the old buffer have reported
            _SNAP_RETIRED.append(buf)
        buf = torch.zeros(max(nbytes // 2, 8), dtype=torch.float16, device=dev)
        _SNAP[key] = buf
        _words(dev)
    return buf


def _words(dev, captured=False):
    """The words that launches on the current stream of `dev` report into (kept when the buffer is outgrown: launches in flight and
    captured HIP graphs hold their address).  captured: for a launch that is being recorded any words of the device will do, it is
    not known where the graph will be replayed, and nothing should be allocated."""
    key = _key(dev)
    if key not in _STATUS:
        for other, words in _STATUS.items():
            if captured and other[0] == key[0]:
                return words
        _STATUS[key] = torch.zeros(2, dtype=torch.int32, pin_memory=True)
    return _STATUS[key]


def _status_word(buf):
    off = L.lib().qt_gdn_chunk_status_offset() // 4
    return buf.view(torch.int32)[off:off + 1]


def _describe(v):
    what = []
    if v & GAVE_UP:
        what.append("an output workgroup waited for its chunk for too long and gave up (its rows were not written)")
    if v & NOT_FINITE:
        what.append("a value is not finite: a half-precision operand overflowed (|state|, |v| or an intermediate above 65504)")
    return "; ".join(what) or f"status {v}"


def _raise_if_failed(keys):
    """Looks at what launches have reported into the pinned host words of `keys`, without waiting (a launch still in flight is judged
    at the next call).  A report is cleared, here and in the buffer's status word, and raised as ChunkedPrefillError."""
    v = 0
    for key in keys:
        pin = _STATUS[key]
        if pin[0] or pin[1]:
            torch.cuda.current_stream(key[0]).synchronize()      # error path only: no launch of this stream may report after the reset
            v |= (GAVE_UP if pin[0] else 0) | (NOT_FINITE if pin[1] else 0)
            if key in _SNAP:
                _status_word(_SNAP[key]).zero_()
            pin.zero_()
    if v:
        raise ChunkedPrefillError("chunked prefill: " + _describe(v))


def _provide_snap(index, nbytes):
    """The buffer of the current stream of device `index` and its report words, for the native launch path (which keeps them until
    it needs a larger one)."""
    dev = torch.device("cuda", index)
    return _snap_buffer(dev, nbytes), _words(dev)


def _provide_words(index):
    return _words(torch.device("cuda", index), captured=True)


def _report_found(index):
    _raise_if_failed([_key(torch.device("cuda", index))])


L.on_host_load(lambda host: host.set_hooks(_provide_snap, _provide_words, _report_found))


def check_status(device=None, sync=True):
    """Raises ChunkedPrefillError if a chunked-prefill launch on `device` has reported a failure, whichever stream it ran on: a
    launch in a replayed HIP graph reports into the words of the stream that it was captured on (or of another one of the device).
    sync: wait for the current stream first.  phase_b / phase_b_norm look at the words of their own stream, without waiting, before
    every launch; a caller that needs the answer for the launches and replays already made calls this on their stream with
    sync=True.  While the current stream is being captured nothing is looked at."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    if torch.cuda.is_current_stream_capturing():
        return
    if sync:
        torch.cuda.current_stream(dev).synchronize()
    _raise_if_failed([key for key in _STATUS if key[0] == _key(dev)[0]])


def phase_b(q, k, v, Tb, Am, gv, state, relaxed=True, flags=DEFAULT_FLAGS, tg=None):
    """The serial state recurrence on the outputs of phase A -> y [S,16,128] bf16, new state [1,16,128,128] f32
    (qwen35/gdn_nax.py:404-410).  Tb / Am / gv are the records prep_a (or gdn_chunked's phase A) produced."""
    return L.host.phase_b(q.shape[0], Tb, Am, gv, state)


def phase_b_norm(proj, Tb, Am, gv, state, gw, eps=1e-6):
    """phase_b followed by prefill.gated_norm (qwen35/prefill.py:241-244) in one pass: the outputs never leave the chip
    un-normalised.  proj [S,8224] bf16 supplies z; gw [128].  -> out [S,2048] bf16, new state [1,16,128,128] f32."""
    return L.host.phase_b_norm(proj, Tb, Am, gv, state, gw, eps)
