"""TTT-MLP memory-cache combiner on the HIP path: the segment loop of
`TTTMLP.ttt` (ttt_layer.py:506-561) as two fused launches per direction
instead of one cached-readout launch per (segment, memo state) pair.

For a token of segment i >= 1 (segments of M mini-batches), with
summary_j = mean of XK over segment j and gamma = softmax_j(XU . summary_j)
over j = 0..i:

    out = gamma_i XQW + sum_{j<i} gamma_j (XQ + LN_1e-6(gelu(XQ W1_j + b1_j) W2_j + b2_j) ln_w + ln_b)

Segment 0 keeps XQW.  The memo states are the `TritonMLP.apply` memo outputs
with the same M.  Gradients flow into XQW, XU and XK, as in the reference: it
runs the cached readouts under `torch.no_grad`, and a segment's summary enters
its own tokens' gates undetached (ttt_layer.py:519,528) but is cached detached
(:521,559), so XK of a segment gets the mean-summary gradient of its own
segment only.  Unlike the reference's cached-readout kernel, every (b,h)
chain uses its own memo states.

Layouts follow the caller (ttt_layer.py:453-561): XQ, XK, XU, XQW
[B,H,NC,K,F]; W1_memo [B,H,NS,F,FF], b1_memo [B,H,NS,1,FF], W2_memo
[B,H,NS,FF,F], b2_memo [B,H,NS,1,F] fp32; LN parameters [H,F]."""

from __future__ import annotations

import math

import torch

from . import _lib
from ._common import as_act, check_device, dtype_code, f32c, grads_as, on_device, ptr, stream_of

READOUT_EPS = 1e-6  # kernels/mlp_cached_readout.py:98


def _check(XQ, XK, XU, XQW, W1, b1, W2, b2, ln_w, ln_b, M):
    if XQ.dim() != 5:
        raise ValueError(f"XQ must be [B,H,NC,K,F], got {tuple(XQ.shape)}")
    B, H, NC, K, F = XQ.shape
    for name, t in (("XK", XK), ("XU", XU), ("XQW", XQW)):
        if tuple(t.shape) != (B, H, NC, K, F):
            raise ValueError(f"{name} shape {tuple(t.shape)} != XQ shape {tuple(XQ.shape)}")
    M = int(M)
    if M < 1:
        raise ValueError(f"memo segment size M must be >= 1, got {M}")
    NS = math.ceil(NC / M)
    FF = W1.shape[-1]
    want = {"W1_memo": (W1, (B, H, NS, F, FF)), "b1_memo": (b1, (B, H, NS, 1, FF)),
            "W2_memo": (W2, (B, H, NS, FF, F)), "b2_memo": (b2, (B, H, NS, 1, F))}
    for name, (t, shp) in want.items():
        if tuple(t.shape) != shp:
            raise ValueError(f"{name} must be {shp}, got {tuple(t.shape)}")
    if tuple(ln_w.shape) != (H, F) or tuple(ln_b.shape) != (H, F):
        raise ValueError(f"LN weight/bias must be [H,F]={(H, F)}")
    return B, H, NC, K, F, FF, M


def memo_combine_forward(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M: int,
                         eps: float = READOUT_EPS, images: bool = True, rows=None):
    """Run the combiner.  Returns (out [B,H,NC,K,F] in XQW.dtype, gates) where
    `gates` (uint8 device buffer) is what memo_combine_backward needs.  With
    `images` (bf16), the workspace also holds each memo state's LDS image,
    written once here and copied straight into LDS by this call and the
    backward: worth its one conversion pass when a backward follows; without
    it every workgroup converts the states it stages (the same results).  `rows`
    (a flat fp32 tensor of memo_rows floats) receives the readouts' centred rows
    and their 1/sigma, from which the backward forms the gate gradients."""
    B, H, NC, K, F, FF, M = _check(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M)
    dev = check_device(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b)
    mp = XQW.dtype
    code = dtype_code(mp)
    xq, xk, xu, xqw = (as_act(t, mp) for t in (XQ, XK, XU, XQW))
    ws = [f32c(t) for t in (W1_memo, b1_memo, W2_memo, b2_memo)]
    lw, lb = f32c(ln_w), f32c(ln_b)
    lib = _lib.load()
    # the gates and, for bf16, the memo states' LDS images that both calls copy in
    nbytes = (lib.ttt_mlp_memo_workspace_bytes(B, H, NC, K, F, FF, M, code) if images
              else lib.ttt_mlp_memo_gates_bytes(B, H, NC, K, F, M))
    gates = torch.empty(nbytes, device=dev, dtype=torch.uint8)
    out = torch.empty((B, H, NC, K, F), device=dev, dtype=mp)
    with on_device(dev):
        args = (ptr(xq), ptr(xk), ptr(xu), ptr(xqw), *(ptr(t) for t in ws), ptr(lw), ptr(lb), B, H, NC, K, F, FF, M,
                code, float(eps), ptr(out), ptr(gates), gates.numel())
        if rows is None:
            st = lib.ttt_mlp_memo_combine(*args, stream_of(dev))
        else:
            st = lib.ttt_mlp_memo_combine_keep(*args, ptr(rows), rows.numel() * 4, stream_of(dev))
    _lib.check(st, "ttt_mlp_memo_combine")
    return out, gates


def memo_combine_backward(XQ, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M: int, gates, dout,
                          eps: float = READOUT_EPS):
    """Gradients (dXK, dXU, dXQW) in XQW.dtype of the combiner run that produced `gates`."""
    B, H, NC, K, F = XQ.shape
    FF = W1_memo.shape[-1]
    dev = check_device(XQ, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, gates, dout)
    mp = XQW.dtype
    code = dtype_code(mp)
    xq, xu, xqw, do = (as_act(t, mp) for t in (XQ, XU, XQW, dout))
    ws = [f32c(t) for t in (W1_memo, b1_memo, W2_memo, b2_memo)]
    lw, lb = f32c(ln_w), f32c(ln_b)
    dxk, dxu, dxqw = (torch.empty((B, H, NC, K, F), device=dev, dtype=mp) for _ in range(3))
    lib = _lib.load()
    with on_device(dev):
        st = lib.ttt_mlp_memo_combine_bwd(ptr(xq), ptr(xu), ptr(xqw), *(ptr(t) for t in ws), ptr(lw), ptr(lb),
                                          ptr(do), B, H, NC, K, F, FF, int(M), code, float(eps), ptr(gates),
                                          gates.numel(), ptr(dxk), ptr(dxu), ptr(dxqw), stream_of(dev))
    _lib.check(st, "ttt_mlp_memo_combine_bwd")
    return dxk, dxu, dxqw


# The kept rows grow with the square of the sequence: past this, the backward
# forms the readouts again.
ROWS_MAX_BYTES = 1 << 30
# Rows of this size stay in the caches on their way to the backward.
ROWS_CACHED_BYTES = 16 << 20


def memo_rows(B: int, H: int, NC: int, K: int, F: int, M: int) -> int:
    """Floats of the readouts' rows that a training forward can keep, 0
    where there are none or they pass ROWS_MAX_BYTES."""
    n = _lib.load().ttt_mlp_memo_rows_bytes(B, H, NC, K, F, M)
    return n // 4 if n <= ROWS_MAX_BYTES else 0


def training_form(rows: int, FF: int, dtype: torch.dtype):
    """(whether a training forward keeps its `rows` floats of rows, whether it
    writes the memo states' images).  A kept row is written and read once instead
    of being formed again, which costs F FF products and FF GELUs: in fp32 the
    rows are the cheaper at every size, in 16 bits from 128 hidden units on, and
    below that only while the caches hold them.  Forward + backward, us, rows formed again (with
    images) / kept without images / kept with images:
      B16 H12 T2048 M8 bf16: F64 FF32 371/533/523, FF64 480/588/549, FF128 654/664/646,
                             FF256 1,018/881/868; F32 FF32 209/264/249, FF64 268/290/276, FF128 400/372/356
      B8 H12 T1024 M2 bf16:  F64 FF64 271/319/281, FF128 399/422/376
      B1 H4 T1024 M8 bf16:   F64 FF64 66/55/56, FF256 104/75/76; F32 FF32 47/44/44
      B16 H12 T2048 M8 fp32: F64 FF32 790/774, FF256 3,704/2,216; F32 FF32 482/424."""
    small = 4 * rows <= ROWS_CACHED_BYTES
    keep = rows > 0 and (dtype == torch.float32 or FF >= 128 or small)
    return keep, not (keep and small)


def memo_combine_backward_kept(XQ, XU, XQW, ln_w, ln_b, M: int, gates, rows, dout):
    """memo_combine_backward from the rows that the forward kept."""
    B, H, NC, K, F = XQ.shape
    dev = check_device(XQ, XU, XQW, ln_w, ln_b, gates, rows, dout)
    mp = XQW.dtype
    xq, xu, xqw, do = (as_act(t, mp) for t in (XQ, XU, XQW, dout))
    lw, lb = f32c(ln_w), f32c(ln_b)
    dxk, dxu, dxqw = (torch.empty((B, H, NC, K, F), device=dev, dtype=mp) for _ in range(3))
    with on_device(dev):
        st = _lib.load().ttt_mlp_memo_combine_bwd_kept(
            ptr(xq), ptr(xu), ptr(xqw), ptr(lw), ptr(lb), ptr(do), B, H, NC, K, F, int(M), dtype_code(mp), ptr(gates),
            gates.numel(), ptr(rows), rows.numel() * 4, ptr(dxk), ptr(dxu), ptr(dxqw), stream_of(dev))
    _lib.check(st, "ttt_mlp_memo_combine_bwd_kept")
    return dxk, dxu, dxqw


class MemoCombineFunction(torch.autograd.Function):
    """apply(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M[, eps]) -> out.
    Differentiable wrt XK, XU and XQW (as the reference's loop is)."""

    @staticmethod
    def forward(ctx, XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M, eps=READOUT_EPS):
        # an inference call writes neither rows nor images
        keep = images = False
        if any(ctx.needs_input_grad[1:4]):
            n = memo_rows(*XQ.shape, int(M)) if XQ.dim() == 5 and int(M) > 0 else 0
            keep, images = training_form(n, W1_memo.shape[-1], XQW.dtype)
        rows = torch.empty(n, device=XQ.device, dtype=torch.float32) if keep else None
        out, gates = memo_combine_forward(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M, eps,
                                          images=images, rows=rows)
        if keep:
            ctx.save_for_backward(XQ, XU, XQW, ln_w, ln_b, gates, rows)
        else:
            ctx.save_for_backward(XQ, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, gates)
        ctx.M, ctx.eps = int(M), eps
        ctx.dtypes = (XK.dtype, XU.dtype, XQW.dtype)
        return out

    @staticmethod
    def backward(ctx, dout):
        saved = ctx.saved_tensors
        if len(saved) == 7:
            XQ, XU, XQW, lw, lb, gates, rows = saved
            dxk, dxu, dxqw = memo_combine_backward_kept(XQ, XU, XQW, lw, lb, ctx.M, gates, rows, dout)
        else:
            XQ, XU, XQW, W1, b1, W2, b2, lw, lb, gates = saved
            dxk, dxu, dxqw = memo_combine_backward(XQ, XU, XQW, W1, b1, W2, b2, lw, lb, ctx.M, gates, dout, ctx.eps)
        return (None,) + grads_as((dxk, dxu, dxqw), ctx.dtypes) + (None,) * 8


def mlp_memo_combine(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, M: int):
    """Drop-in for the segment loop of TTTMLP.ttt (ttt_layer.py:506-561): given
    the TritonMLP.apply output XQW_batch and memo, returns the combined
    XQW_batch [B,H,NC,K,F] (before the caller's permute/reshape)."""
    return MemoCombineFunction.apply(XQ, XK, XU, XQW, W1_memo, b1_memo, W2_memo, b2_memo, ln_w, ln_b, int(M))


__all__ = ["mlp_memo_combine", "MemoCombineFunction", "memo_combine_forward", "memo_combine_backward"]
