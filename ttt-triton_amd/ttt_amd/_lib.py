"""ctypes binding of libttt_amd.so (declared in include/ttt_amd.h).

The library is loaded from this directory.  There is no fallback: if the
library is missing or fails to load, every entry point raises."""

from __future__ import annotations

import ctypes
import functools
import os
import threading

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
# TTT_AMD_LIB names another build of the same library (e.g. the host-ASan
# checking build of build_lib.py --asan)
LIB_PATH = os.environ.get("TTT_AMD_LIB") or os.path.join(_HERE, "libttt_amd.so")
ABI_VERSION = 11

DTYPE_F32 = 0
DTYPE_BF16 = 1
DTYPE_F16 = 2

# eta forms (enum ttt_eta_rule): the dense [B,H,NC,K,K] tensor, or the per-token
# learning rate lr [B,H,NC,K] fp32 expanded on chip by a rule
ETA_DENSE = 0
ETA_LAYER = 1
ETA_CAUSAL = 2
ETA_DENSE_F32 = 3  # dense eta kept in fp32 under 16-bit activations (chosen from eta's dtype)
FORM_SPLIT = 0x100  # or'ed into the eta rule: the state and the readout as two launches
STATE_SHARED = 0x200  # (forward): initial states [H,...], one for every sequence
SAVED_SLOTS = 0x400  # `saved` without the place of the backward's handoff (slot_saved below)
ETA_RULES = {"dense": ETA_DENSE, "layer": ETA_LAYER, "causal": ETA_CAUSAL}

# process-wide options (enum ttt_option)
OPT_MLP_BWD_POLL_LIMIT = 1
OPT_MLP_BWD_FUSED = 2
OPT_SMALL_KERNELS = 3

STATUS_TIMEOUT = -8
STATUS_SCRATCH = -9
MLP_BWD_NOALLOC_SCRATCH_BYTES = 64 << 20

_P = ctypes.c_void_p
_I = ctypes.c_int
_F = ctypes.c_float
_S = ctypes.c_size_t

# name -> (restype, argtypes); mirrors include/ttt_amd.h
SIGNATURES = {
    "ttt_abi_version": (_I, []),
    "ttt_error_string": (ctypes.c_char_p, [_I]),
    "ttt_linear_fwd": (_I, [_P] * 8 + [_I] * 8 + [_F] + [_P] * 5 + [_P, _S, _P]),
    "ttt_linear_saved_bytes": (_S, [_I] * 5),
    "ttt_linear_bwd": (_I, [_P] * 9 + [_I] * 8 + [_F] + [_P] * 8 + [_P, _S, _P]),
    "ttt_linear_bwd_ws": (_I, [_P] * 9 + [_I] * 8 + [_F] + [_P] * 8 + [_P, _S, _P, _S, _P]),
    "ttt_mlp_fwd": (_I, [_P] * 10 + [_I] * 10 + [_F] + [_P] * 13 + [_P, _S, _P]),
    "ttt_mlp_saved_bytes": (_S, [_I] * 7),
    "ttt_split_saved_bytes": (_S, [_I] * 6),
    "ttt_slots_bytes": (_S, [_I] * 7),
    "ttt_mlp_bwd_workspace_bytes": (_S, [_I] * 7),
    "ttt_mlp_bwd": (_I, [_P] * 15 + [_I] * 9 + [_F] + [_P] * 10 + [_P, _S, _P, _S, _P]),
    "ttt_mlp_bwd_noalloc": (_I, [_P] * 15 + [_I] * 9 + [_F] + [_P] * 10 + [_P, _S, _P]),
    "ttt_set_option": (_I, [_I, ctypes.c_longlong]),
    "ttt_get_option": (ctypes.c_longlong, [_I]),
    "ttt_mlp_bwd_check": (_I, [_P, _S] + [_I] * 7 + [_P]),
    "ttt_layer_io_partial_bytes": (_S, [_I] * 4),
    "ttt_qkvu_producer_fwd": (_I, [_P, _I] + [_P] * 3 + [_I] * 5 + [_F, _F, _I] + [_P] * 5 + [_P]),
    "ttt_qkvu_producer_bwd": (_I, [_P, _I] + [_P] * 3 + [_P] * 5 + [_I] * 5 + [_F, _F, _I] + [_P, _P, _S, _P]),
    "ttt_post_norm_fwd": (_I, [_P] * 3 + [_I] * 5 + [_F, _I] + [_P, _P, _P]),
    "ttt_post_norm_bwd": (_I, [_P] * 4 + [_I] * 6 + [_P, _P, _S, _P]),
    "ttt_mlp_cached_readout": (_I, [_P] * 7 + [_I] * 8 + [_F] + [_P, _P]),
    "ttt_mlp_memo_gates_bytes": (_S, [_I] * 6),
    "ttt_mlp_memo_workspace_bytes": (_S, [_I] * 8),
    "ttt_mlp_memo_combine": (_I, [_P] * 10 + [_I] * 8 + [_F] + [_P, _P, _S, _P]),
    "ttt_mlp_memo_rows_bytes": (_S, [_I] * 6),
    "ttt_mlp_memo_combine_keep": (_I, [_P] * 10 + [_I] * 8 + [_F] + [_P, _P, _S, _P, _S, _P]),
    "ttt_mlp_memo_combine_bwd_kept": (_I, [_P] * 6 + [_I] * 7 + [_P, _S, _P, _S] + [_P] * 4),
    "ttt_mlp_memo_combine_bwd": (_I, [_P] * 10 + [_I] * 8 + [_F] + [_P, _S, _P, _P, _P, _P]),
}

_lock = threading.Lock()
_lib = None


class TTTError(RuntimeError):
    pass


def load(path: str = LIB_PATH):
    """Load (once) and return the ctypes library handle."""
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(path):
            raise TTTError(f"{path} not found: build it with `python ttt-triton_amd/build_lib.py`")
        lib = ctypes.CDLL(path)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        v = lib.ttt_abi_version()
        if v != ABI_VERSION:
            raise TTTError(f"libttt_amd ABI version {v}, expected {ABI_VERSION}")
        _lib = lib
        return lib


def check(status: int, what: str) -> None:
    if status != 0:
        msg = load().ttt_error_string(status).decode()
        if status in (-5, STATUS_TIMEOUT):
            raise TTTError(f"{what}: {msg}")
        raise ValueError(f"{what}: {msg} (status {status})")


def fast_linear_shape(K: int, F: int) -> bool:
    """Shapes of the specialised TTT-Linear kernels (16-token mini-batches in
    registers); every other valid shape takes the general-shape kernels, whose
    forward needs the saved buffer as scratch even without a backward."""
    return K == 16 and F in (32, 64)


def fast_mlp_shape(K: int, F: int, FF: int) -> bool:
    return fast_linear_shape(K, F) and FF in (64, 128, 256)


# A training forward's `saved` has the place of the backward's handoff up to this
# size; past it, and in inference, it holds the slots alone, and the backward
# copies them into a buffer of its own first.
SLOTS_WITH_HANDOFF_BYTES = 1 << 30


@functools.lru_cache(maxsize=1024)
def slot_bytes(B: int, H: int, NC: int, K: int, F: int, FF: int, split: bool):
    """Where a mini-batch has a slot (FF = 0: the Linear loop): the bytes of `saved`
    with the place of the handoff, and of the slots alone; 0 elsewhere."""
    lib = load()
    slots = lib.ttt_slots_bytes(B, H, NC, K, F, FF, split)
    if not slots:
        return 0, 0
    full = (lib.ttt_split_saved_bytes(B, H, NC, K, F, FF) if split else
            lib.ttt_mlp_saved_bytes(B, H, NC, K, F, FF, 0) if FF else lib.ttt_linear_saved_bytes(B, H, NC, K, F))
    return full, slots


def slot_saved(*shape_split, train: bool):
    """(bytes of `saved`, SAVED_SLOTS or 0) of a forward, (0, 0) where no mini-batch has a slot."""
    full, slots = slot_bytes(*shape_split)
    return (slots, SAVED_SLOTS if slots else 0) if not train or full > SLOTS_WITH_HANDOFF_BYTES else (full, 0)


def slot_workspace(saved, *shape_split):
    """(bytes of the backward's workspace, SAVED_SLOTS or 0) given the forward's `saved`."""
    full, slots = slot_bytes(*shape_split)
    return (full, SAVED_SLOTS) if slots and saved.numel() == slots else (0, 0)


# The split form's `saved` is bounded: it holds every mini-batch's state.
SPLIT_MAX_BYTES = 1 << 30


def split_form(XQ, FF: int, train: bool = True) -> bool:
    """Whether 16-token mini-batches in fp32 run the split form (FORM_SPLIT; FF = 0:
    the Linear loop).  One chain is one workgroup of the specialised kernels,
    whose readout shares that workgroup's time with the recurrence; the split
    form runs it on the rest of the GPU, and loses once the chains fill that, or
    where there is hardly a recurrence to run beside.  Specialised / split, us in a
    captured graph, forward + backward at 8, 64, 128 (MLP, F = 64, FF = 256: 8, 32)
    chains of 32 mini-batches, then the forward alone:
      Linear       349/197, 356/242, 356/329    126/64, 128/79, 128/94
      MLP 64/64    559/384, 568/462             185/139, 187/161
      MLP 32/128   757/483, 765/571             279/155, 281/180
      MLP 64/256   1,239/946, 1,249/1,118       434/304, 436/329
    Short sequences, forward + backward (chains):
      1 mini-batch: Linear 36/26 (8), MLP 64/64 41/40 (64), 32/128 49/46 (64), 64/256 67/80 (1)
      2, 3:         MLP 64/256 114/121, 155/149 (32)
    and the forward alone:
      Linear       1 mini-batch 12/19 (1), 2: 16/19 (1), 3: 20/18 (64), 4: 23/20 (64)
      MLP 64/64    2: 19/22 (8), 3: 25/25 (8) 25/29 (64), 4: 30/32 (32) 30/34 (64), 6: 41/40 (32), 8: 53/55 (64)
      MLP 64/256   2: 36/40 (8), 3: 50/49 (8) 50/54 (32), 4: 63/64 (32), 6: 90/81 (32)
      MLP 32/128   2: 25/27 (64), 3: 33/32 (64)
    so the forward alone takes 3 mini-batches, and of the 64-wide MLPs at most 6
    chains for each; a forward with a backward behind it, of the MLP 64/256, takes 3.
    In 16 bits the specialised kernels' shorter products win at every count."""
    if XQ.dim() != 5 or XQ.dtype != torch.float32:
        return False
    B, H, NC, K, F = XQ.shape
    if NC < 3 and (FF == 256 or not train):
        return False
    most = 32 if FF == 256 else 64 if FF else 128
    if not train and FF and F == 64:
        most = min(most, 6 * NC)
    if B * H > most:
        return False
    return 0 < slot_bytes(B, H, NC, K, F, FF, True)[0] <= SPLIT_MAX_BYTES


def eta_rule_code(rule) -> int:
    """ttt_eta_rule code of `rule` ("dense", "layer", "causal" or the code)."""
    if isinstance(rule, str):
        if rule not in ETA_RULES:
            raise ValueError(f"unknown eta rule {rule!r} (dense, layer or causal)")
        return ETA_RULES[rule]
    if int(rule) not in ETA_RULES.values():
        raise ValueError(f"unknown eta rule {rule}")
    return int(rule)


def set_option(option: int, value: int) -> None:
    check(load().ttt_set_option(int(option), int(value)), "ttt_set_option")


def get_option(option: int) -> int:
    return int(load().ttt_get_option(int(option)))
