"""The buffers of the kernels that keep a slot per mini-batch (csrc/ttt_wide.h):
what a forward needs, the backward's handoff beside or behind it, and the size
past which the general-shape kernels run."""

import os
import subprocess

import pytest
import torch

from tests._util import rel_l2, to_dev
from tests.test_gpu_wide import LIN_KEYS, MLP_KEYS, _inputs

F32, BF16 = torch.float32, torch.bfloat16
SHAPES = [(32, 64, 0), (48, 64, 0), (64, 64, 64), (64, 64, 256), (48, 32, 128)]  # K, F, FF (0: Linear)
SPLIT = [(16, 64, 0), (16, 64, 256), (16, 32, 128)]
LIMIT = 4 << 30


def _sizes(K, F_, FF):
    """Floats of a state, of a mini-batch's forward values and of its handoff."""
    if FF:
        return 2 * F_ * FF + FF + F_, 2 * K * (FF + F_) + K, 2 * F_ * FF + FF + F_ + 2 * K * (FF + F_) + 2 * F_ + K
    return F_ * F_ + F_, 2 * K * F_ + K, F_ * F_ + F_ + 2 * K * F_ + 2 * F_ + K


def test_layout(tmp_path):
    """Which wave reads which token's eta (never past the mini-batch), the slot's
    parts, alignment, LDS size: csrc/ttt_wide_layout.h enumerated on the host."""
    here = os.path.dirname(os.path.abspath(__file__))
    csrc = os.path.join(os.path.dirname(here), "ttt-triton_amd", "csrc")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, os.path.join(here, "wide_layout_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert (r.returncode, r.stdout) == (0, "16\n"), r.stdout


@pytest.mark.parametrize("split,shape", [(0, s) for s in SHAPES] + [(1, s) for s in SPLIT])
def test_bytes(split, shape):
    from ttt_amd import _lib
    lib = _lib.load()
    K, F_, FF = shape
    B, H, NC = 3, 5, 7
    state, values, hand = _sizes(*shape)
    n = B * H * NC
    assert lib.ttt_slots_bytes(B, H, NC, K, F_, FF, split) == 4 * (n * (state + values) + B * H * state)
    full = (lib.ttt_split_saved_bytes(B, H, NC, K, F_, FF) if split else lib.ttt_mlp_saved_bytes(B, H, NC, K, F_, FF, 1)
            if FF else lib.ttt_linear_saved_bytes(B, H, NC, K, F_))
    assert full == 4 * n * (state + values + hand)
    for other in ((16, 64, FF) if not split else (32, F_, FF), (K, 48, FF)):
        assert lib.ttt_slots_bytes(B, H, NC, *other, split) == 0


@pytest.mark.parametrize("K,F_,FF", SHAPES)
def test_past_the_limit_the_general_layout(K, F_, FF):
    from ttt_amd import _lib
    lib = _lib.load()
    state, values, hand = _sizes(K, F_, FF)
    H = 64
    NC = LIMIT // (4 * H * (state + values))
    saved = lambda nc: (lib.ttt_mlp_saved_bytes(1, H, nc, K, F_, FF, 1) if FF  # noqa: E731
                        else lib.ttt_linear_saved_bytes(1, H, nc, K, F_))
    assert lib.ttt_slots_bytes(1, H, NC, K, F_, FF, 0) > 0 == lib.ttt_slots_bytes(1, H, NC + 1, K, F_, FF, 0)
    assert saved(NC) == 4 * H * NC * (state + values + hand)
    # the states and one mini-batch's scratch per chain
    assert 4 * H * NC * state < saved(NC + 1) < 4 * H * NC * state + H * (32 << 20) < saved(NC)


def test_validation():
    from ttt_amd import _lib
    lib = _lib.load()
    P, SLOTS, SPLIT_ = 0x10000, _lib.SAVED_SLOTS, _lib.FORM_SPLIT

    def fwd(nbytes, K=64, F_=64, rule=SLOTS):
        return lib.ttt_linear_fwd(*([P] * 8), 2, 4, 8, K, F_, 4, 0, rule, 1e-8, P, None, None, None, None, P, nbytes, None)

    def bwd(nbytes, ws, wbytes, K=64, rule=SLOTS):
        return lib.ttt_linear_bwd_ws(*([P] * 9), 2, 4, 8, K, 64, 4, 0, rule, 1e-8, *([P] * 8), P, nbytes, ws, wbytes, None)

    for K, split in ((64, 0), (16, SPLIT_)):
        full, slots = _lib.slot_bytes(2, 4, 8, K, 64, 0, bool(split))
        assert fwd(slots - 4, K, rule=SLOTS | split) == -6 == fwd(slots, K, rule=split)
        assert bwd(slots - 4, P, full, K, SLOTS | split) == -6 == bwd(slots, None, full, K, SLOTS | split)
        assert bwd(slots, P, full - 4, K, SLOTS | split) == -6 and bwd(slots, P + 8, full, K, SLOTS | split) == -4
        assert bwd(slots, P, full, K, split) == -6  # (a forward with the handoff's place)
    assert fwd(1 << 40, 32, 48) == fwd(1 << 40, 16, 64) == -7  # no such slots
    args = [P] * 15 + [2, 4, 8, 64, 64, 64, 4, 0, SLOTS, 1e-8] + [P] * 10
    assert lib.ttt_mlp_bwd(*args, P, lib.ttt_slots_bytes(2, 4, 8, 64, 64, 64, 0), P, 256, None) == -6


def test_which_forwards_take_the_slots_alone(monkeypatch):
    from ttt_amd import _lib
    shape = (2, 3, 5, 64, 64, 64, False)
    full, slots = _lib.slot_bytes(*shape)
    assert 0 < slots < full
    assert _lib.slot_saved(*shape, train=False) == (slots, _lib.SAVED_SLOTS)
    for bound, got in ((full, (full, 0)), (full - 1, (slots, _lib.SAVED_SLOTS))):
        monkeypatch.setattr(_lib, "SLOTS_WITH_HANDOFF_BYTES", bound)
        assert _lib.slot_saved(*shape, train=True) == got
    assert _lib.slot_saved(2, 3, 5, 32, 48, 48, False, train=True) == (0, 0)
    x = lambda n: torch.empty(n, dtype=torch.uint8, device="meta")  # noqa: E731
    assert _lib.slot_workspace(x(slots), *shape) == (full, _lib.SAVED_SLOTS)
    assert _lib.slot_workspace(x(full), *shape) == (0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("split,K,F_,FF,dt", [(0, *s, dt) for s in SHAPES for dt in (F32, BF16)] +
                         [(1, *s, F32) for s in SPLIT])
def test_with_the_handoffs_place_and_without(monkeypatch, split, K, F_, FF, dt):
    """The same outputs and gradients, bitwise, from either `saved`, and
    of a second backward, which leaves the slots as they were."""
    from ttt_amd import _lib
    from ttt_amd.linear import linear_backward, linear_forward
    from ttt_amd.mlp import mlp_backward, mlp_forward
    B, H, NC, G = 2, 3, 5, 2
    g = to_dev(_inputs(B, H, NC, K, F_, FF, dt, "layer", K + FF))
    full, slots = _lib.slot_bytes(B, H, NC, K, F_, FF, bool(split))
    kw = dict(want_last=True, want_saved=True, split=bool(split))
    res = []
    for bound, size in ((full, full), (0, slots)):
        monkeypatch.setattr(_lib, "SLOTS_WITH_HANDOFF_BYTES", bound)
        if FF:
            out, ck, _, last, saved = mlp_forward(*(g[k] for k in MLP_KEYS), G, **kw)
        else:
            out, ck, last, saved = linear_forward(*(g[k] for k in LIN_KEYS), G, **kw)
        assert saved.numel() == size
        kept = saved.clone()
        for _ in range(2):
            head = (g["ln_w"], g["ln_b"], g["XQ"], g["XV"], g["XK"], g["eta"])
            if FF:
                a, b = mlp_backward(*head, None if split else ck, None if split else last, saved, g["dOut"], G, FF=FF)
            else:
                a, b = linear_backward(*head, None if split else ck[0], None if split else last[0], saved, g["dOut"], G,
                                       split=bool(split))
            res.append([out, *last, *a, *b])
    assert torch.equal(saved, kept)
    for got in res[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got, res[0]))


@pytest.mark.gpu
def test_past_the_limit_on_the_gpu():
    """A call whose slots pass the limit runs, on the general-shape kernels: its
    first chains agree with the same chains alone, on the slots' kernels."""
    from ttt_amd import _lib
    from ttt_amd.linear import TTTLinearFunction
    B, NC, K, F_ = 1024, 127, 32, 64
    lib = _lib.load()
    assert lib.ttt_slots_bytes(B, 1, NC, K, F_, 0, 0) == 0 < lib.ttt_slots_bytes(2, 1, NC, K, F_, 0, 0)
    gen = torch.Generator(device="cuda").manual_seed(0)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    x = [torch.nn.functional.normalize(r(B, 1, NC, K, F_), dim=-1).to(BF16) for _ in range(3)]
    lr = 0.1 * torch.sigmoid(r(B, 1, NC, K)) / F_
    ln, ws = [1 + 0.1 * r(1, F_), 0.1 * r(1, F_)], [0.02 * r(B, 1, F_, F_), 0.02 * r(B, 1, 1, F_)]
    dout = r(B, 1, NC, K, F_).to(BF16)
    res = []
    for b in (B, 2):
        leaf = [t[:b].detach().requires_grad_(True) for t in (*ws, *x, lr)]
        out = TTTLinearFunction.apply(*ln, *leaf, 8, 1e-8, "layer")
        res.append([out.detach()[:2], *(t[:2] for t in torch.autograd.grad(out, leaf, dout[:b]))])
    for a, b in zip(*res):
        # (fp32 sums in another order; bf16 values at a rounding boundary)
        assert rel_l2(a, b) <= (1e-4 if a.dtype == F32 else 2e-3)
