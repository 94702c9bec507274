"""Small host-side helpers shared by the launchers."""

from __future__ import annotations

import contextlib

import torch

from . import _lib


def dtype_code(dt: torch.dtype) -> int:
    if dt == torch.bfloat16:
        return _lib.DTYPE_BF16
    if dt == torch.float16:
        return _lib.DTYPE_F16
    if dt == torch.float32:
        return _lib.DTYPE_F32
    raise ValueError(f"unsupported activation dtype {dt} (float32, bfloat16 or float16)")


def as_act(t: torch.Tensor, dt: torch.dtype) -> torch.Tensor:
    """Activation in the path's dtype, contiguous (no copy when already so)."""
    return t if t.dtype == dt and t.is_contiguous() else t.detach().to(dt).contiguous()


def f32c(t: torch.Tensor) -> torch.Tensor:
    """fp32 and contiguous (no copy when already so)."""
    return as_act(t, torch.float32)


def states(ts):
    """(initial fast weights as the kernels read them, STATE_SHARED or 0): a batch
    expanded from one state ([H,...] with batch stride 0, as the layer passes it)
    is read in place, anything else as a contiguous fp32 [B,H,...]."""
    if all(t.dtype == torch.float32 and t.stride() == (0, t.shape[2] * t.shape[3], t.shape[3], 1)
           and ptr(t) % 16 == 0 for t in ts):
        return ts, _lib.STATE_SHARED
    return [f32c(t) for t in ts], 0


def eta_operand(eta: torch.Tensor, rule: int, dt: torch.dtype):
    """(eta as the kernels read it, the rule code to pass).  A dense eta keeps
    its own dtype when that is fp32 under 16-bit activations (TTT_ETA_DENSE_F32,
    its gradient then fp32 too), as the reference's kernels read eta in
    whatever dtype it comes; any other dense eta goes in the activation dtype.
    A learning-rate vector is fp32."""
    if rule == _lib.ETA_DENSE:
        if eta.dtype == torch.float32 and dt != torch.float32:
            return f32c(eta), _lib.ETA_DENSE_F32
        return as_act(eta, dt), rule
    return f32c(eta), rule


def check_device(*ts: torch.Tensor) -> torch.device:
    dev = ts[0].device
    if dev.type != "cuda":
        raise ValueError("the TTT HIP path needs GPU tensors (device 'cuda')")
    for t in ts[1:]:
        if t.device != dev:
            raise ValueError(f"all tensors must be on {dev}, got {t.device}")
    return dev


_HERE = contextlib.nullcontext()


def on_device(dev: torch.device):
    """torch.cuda.device(dev), free where dev is the current device already."""
    return _HERE if torch.cuda.current_device() == dev.index else torch.cuda.device(dev)


def grads_as(grads, dtypes):
    """Each gradient in its input's type."""
    return tuple(g if g.dtype == dt else g.to(dt) for g, dt in zip(grads, dtypes))


def ptr(t: torch.Tensor) -> int:
    return t.data_ptr()


def stream_of(dev: torch.device) -> int:
    return torch.cuda.current_stream(dev).cuda_stream
