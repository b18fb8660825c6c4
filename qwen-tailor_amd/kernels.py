"""kernels.deltanet: the fused decode / verify GatedDeltaNet step for one sequence (qwen35/kernels.py:555-567);
kernels.fused_gemv: the projections either side of the core (qwen35/kernels.py:291-319)."""
from __future__ import annotations

from . import _lib as L

HV, DK, DV, CD, PW = 16, 128, 128, 6144, 8224


def deltanet(proj, conv_snap, conv_w, A_log, dt_bias, ssm_snap, sel, rows_per_wg: int = 0):
    """proj [M, 8224] bf16 (qkv 6144 | z 2048 | b 16 | a 16 per token).
    conv_snap [S,3,6144] / ssm_snap [S,16,128,128]: state snapshots; the step starts from snapshot sel[0].
    Returns y [M,2048], conv snapshots [M,3,6144] (after each token), ssm snapshots [M,16,128,128]."""
    return L.host.deltanet(proj, conv_snap, conv_w, A_log, dt_bias, ssm_snap, sel, rows_per_wg)


def rms_rows(x, nw, eps=1e-6, T=None, f32=False):
    """The rms prologue of fused_gemv as its own kernel (qwen35/batch.py:295-301): x [M, K] bf16, nw [K] bf16 ->
    BF(nw * (x * rsqrt(mean(x^2) + eps))) [M, K].  T (the reference's threadgroup size) does not change the result and is
    ignored.  f32=True returns the same bf16 values widened to float32, as the reference does."""
    return L.host.rms_rows(x, nw, eps, f32)


def fused_gemv(W, x, *, nw=None, eps=1e-6, res=None, swiglu=False, gnorm=None, T=None, R=None, mtmax=None, wf=False):
    """y = W @ f(x) (qwen35/kernels.py:291-319).  W [N, K] bf16; x [..., K] bf16, or float32 holding bf16 values (what
    rms_rows(f32=True) returns).  nw: rms prologue weight [K]; gnorm = (proj [M, 8224], gw [128]): gated-norm prologue
    (K = 2048); res [..., N]: residual added after rounding the product to bf16; swiglu: rows of W interleave gate and up,
    the result is [..., N/2].  T, R, mtmax, wf are the reference's tilings: they never change its arithmetic and are ignored.
    Weights in the reference's lossless 12-bit form are not taken: pass the plain bf16 matrix."""
    return L.host.fused_gemv(W, x, nw, eps, res, swiglu, gnorm)
