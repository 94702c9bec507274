"""The split form of 16-token mini-batches (TTT_FORM_SPLIT: the state and the
readout as two launches, csrc/ttt_wide.h) against the CPU oracle and the
specialised kernels, and the rule that chooses it.

Tolerances as for the other kernels: fp32 max-abs <= 1e-4, or 8 times the fp32
oracle's own error against fp64 (tests/_util.fp32_bound)."""

import pytest
import torch

from oracle import ttt_oracle as O
from tests._util import oracle_linear_grads, oracle_mlp_grads, rel_l2, to_dev
from tests.test_gpu_wide import LIN_KEYS, MLP_KEYS, SIZES, _check, _inputs

F32 = torch.float32


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["causal", "layer"])
@pytest.mark.parametrize("F_,FF", [(64, 64), (64, 256), (32, 128)])
def test_mlp(F_, FF, kind):
    dt = F32
    from ttt_amd.mlp import mlp_backward, mlp_forward
    for B, H, NC, G, M in SIZES:
        d = _inputs(B, H, NC, 16, F_, FF, dt, kind, F_ + FF + NC)
        g = to_dev(d)
        out, ck, memo, last, saved = mlp_forward(*(g[k] for k in MLP_KEYS), G, M=M, want_ckpt=True, want_last=True,
                                                 split=True)
        (dlw, dlb, dW1, db1, dW2, db2), (dxq, dxv, dxk, deta) = mlp_backward(
            g["ln_w"], g["ln_b"], g["XQ"], g["XV"], g["XK"], g["eta"], None, None, saved, g["dOut"], G, FF=FF)
        torch.cuda.synchronize()
        mine = {"out": out}
        for i, nm in enumerate(("W1", "b1", "W2", "b2")):
            mine.update({nm + "_last": last[i], nm + "_ckpt": ck[i], nm + "_memo": memo[i]})
        full = [O.mlp_forward_full(*(d[k].to(t) for k in MLP_KEYS), G=G, M=M) for t in (torch.float64, F32)]
        _check(mine, *full, dt)
        grads = [oracle_mlp_grads(d, d["dOut"], G=0, dtype=t) for t in (torch.float64, F32)]
        _check(dict(dXQ=dxq, dXV=dxv, dXK=dxk, deta=deta, dW1=dW1, db1=db1, dW2=dW2, db2=db2, dln_w=dlw, dln_b=dlb),
               *grads, dt)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["causal", "layer"])
def test_linear(kind):
    dt = F32
    from ttt_amd.linear import linear_backward, linear_forward
    for B, H, NC, G, _ in SIZES:
        d = _inputs(B, H, NC, 16, 64, 0, dt, kind, NC)
        g = to_dev(d)
        out, ck, last, saved = linear_forward(*(g[k] for k in LIN_KEYS), G, want_ckpt=True, want_last=True, split=True)
        (dlw, dlb, dW1, db1), (dxq, dxv, dxk, deta) = linear_backward(
            g["ln_w"], g["ln_b"], g["XQ"], g["XV"], g["XK"], g["eta"], None, None, saved, g["dOut"], G, split=True)
        torch.cuda.synchronize()
        full = [O.linear_forward_full(*(d[k].to(t) for k in LIN_KEYS), G=G) for t in (torch.float64, F32)]
        _check({"out": out, "W1_last": last[0], "b1_last": last[1], "W1_ckpt": ck[0], "b1_ckpt": ck[1]}, *full, dt)
        grads = [oracle_linear_grads(d, d["dOut"], G=0, dtype=t) for t in (torch.float64, F32)]
        _check(dict(dXQ=dxq, dXV=dxv, dXK=dxk, deta=deta, dW1=dW1, db1=db1, dln_w=dlw, dln_b=dlb), *grads, dt)


@pytest.mark.gpu
@pytest.mark.parametrize("rule", ["dense", "layer", "causal"])
@pytest.mark.parametrize("F_,FF", [(64, 0), (64, 64), (64, 256), (32, 128)])
def test_matches_the_specialised_kernels(F_, FF, rule):
    """Through the autograd Functions on both sides of the rule's chain count,
    a non-contiguous query among the inputs: a batch just past it takes the
    specialised kernels, its first sequences alone the split form."""
    from ttt_amd import _lib
    from ttt_amd.linear import TTTLinearFunction
    from ttt_amd.mlp import TTTMLPFunction
    H, NC, n = 1, 3, 5
    B = (32 if FF == 256 else 64 if FF else 128) + 1
    d = _inputs(B, H, NC, 16, F_, FF, F32, "causal", 3 * F_ + FF)
    keys, fn = (MLP_KEYS, TTTMLPFunction) if FF else (LIN_KEYS, TTTLinearFunction)
    lr = torch.rand(B, H, NC, 16, generator=torch.Generator().manual_seed(F_)) / F_
    res = []
    for b in (B, n):
        g = to_dev({k: v if k in ("ln_w", "ln_b") else v[:b] for k, v in d.items()})
        g["eta"] = g["eta"] if rule == "dense" else lr[:b].cuda()
        # (the strides of a [B, NC, K, H, F] tensor)
        g["XQ"] = g["XQ"].permute(0, 2, 3, 1, 4).contiguous().permute(0, 3, 1, 2, 4)
        assert _lib.split_form(g["XQ"], FF) == (b == n)
        leaf = {k: g[k].detach().requires_grad_(True) for k in keys}
        out = fn.apply(*(leaf[k] for k in keys), 2, *((2,) if FF else ()), O.LN_EPS, rule)
        out, memo = (out[0], out[1:]) if FF else (out, ())
        grads = torch.autograd.grad(out, [leaf[k] for k in keys if k not in ("ln_w", "ln_b")], g["dOut"])
        res.append([out, *memo, *grads])
        with torch.no_grad():
            alone = fn.apply(*(leaf[k] for k in keys), 2, *((2,) if FF else ()), O.LN_EPS, rule)
        assert torch.equal(alone[0] if FF else alone, out)
    torch.cuda.synchronize()
    for a, b in zip(*res):
        assert a.dtype == b.dtype == F32
        # sums in another order, through NC = 3 updates
        assert rel_l2(b, a[:n]) <= 2e-5


def test_rule():
    """fp32, 16-token mini-batches, the kernels' shapes, few chains, a bounded buffer."""
    from ttt_amd import _lib
    x = lambda *s, dt=F32: torch.empty(s, dtype=dt, device="meta")  # noqa: E731
    assert _lib.split_form(x(2, 4, 16, 16, 64), 0) and _lib.split_form(x(2, 4, 16, 16, 32), 128)
    assert _lib.split_form(x(1, 64, 8, 16, 64), 64) and not _lib.split_form(x(1, 65, 8, 16, 64), 64)
    assert _lib.split_form(x(2, 64, 8, 16, 64), 0) and not _lib.split_form(x(2, 65, 8, 16, 64), 0)
    assert _lib.split_form(x(1, 32, 8, 16, 64), 256)
    for dt in (torch.bfloat16, torch.float16):
        assert not _lib.split_form(x(2, 4, 16, 16, 64, dt=dt), 0)
    for shape, FF in (((2, 4, 16, 32, 64), 0), ((2, 4, 16, 16, 32), 0), ((1, 33, 16, 16, 64), 256),
                      ((2, 4, 16, 16, 64), 128), ((0, 4, 16, 16, 64), 0), ((2, 4, 16, 64), 0)):
        assert not _lib.split_form(x(*shape), FF), (shape, FF)
    lib = _lib.load()
    per = lib.ttt_split_saved_bytes(1, 1, 1, 16, 64, 0)
    nc = _lib.SPLIT_MAX_BYTES // per
    assert _lib.split_form(x(1, 1, nc, 16, 64), 0) and not _lib.split_form(x(1, 1, nc + 1, 16, 64), 0)


def test_rule_of_short_sequences():
    """Without a backward from 3 mini-batches on, the 64-wide MLPs with at most 6
    chains for each; with one, the MLP of 256 units from 3 on."""
    from ttt_amd import _lib
    x = lambda *s: torch.empty(s, dtype=F32, device="meta")  # noqa: E731
    for F_, FF in ((64, 0), (64, 64), (64, 256), (32, 128)):
        for NC in (1, 2):
            assert not _lib.split_form(x(1, 1, NC, 16, F_), FF, train=False)
            assert _lib.split_form(x(1, 1, NC, 16, F_), FF) == (FF != 256)
        assert _lib.split_form(x(2, 4, 3, 16, F_), FF) and _lib.split_form(x(2, 4, 3, 16, F_), FF, train=False)
    assert _lib.split_form(x(2, 64, 3, 16, 64), 0, train=False) and _lib.split_form(x(1, 64, 3, 16, 32), 128, train=False)
    for FF, most in ((64, 64), (256, 32)):
        for NC in (3, 4, 5, 16):
            n = min(6 * NC, most)
            assert _lib.split_form(x(1, n, NC, 16, 64), FF, train=False)
            assert not _lib.split_form(x(1, n + 1, NC, 16, 64), FF, train=False)
            assert _lib.split_form(x(1, most, NC, 16, 64), FF)


@pytest.mark.gpu
@pytest.mark.parametrize("F_,FF", [(64, 0), (64, 256)])
def test_inference_allocates_the_slots_alone(F_, FF):
    """No handoff, no gradient buffers: `saved` is what a forward alone needs."""
    from ttt_amd import _lib
    from ttt_amd.linear import linear_forward
    from ttt_amd.mlp import mlp_forward
    B, H, NC = 2, 3, 5
    g = to_dev(_inputs(B, H, NC, 16, F_, FF, F32, "layer", 7))
    res = []
    for want in (False, True):
        r = (mlp_forward(*(g[k] for k in MLP_KEYS), 2, want_saved=want, split=True) if FF else
             linear_forward(*(g[k] for k in LIN_KEYS), 2, want_saved=want, split=True))
        full, slots = _lib.slot_bytes(B, H, NC, 16, F_, FF, True)
        assert r[-1].numel() == (full if want else slots)
        res.append(r[0])
    assert torch.equal(*res)


def test_abi_refuses_what_the_split_form_does_not_take():
    from ttt_amd import _lib
    lib = _lib.load()
    P = 0x10000
    rule = _lib.ETA_DENSE | _lib.FORM_SPLIT

    def fwd(dtype=0, K=16, F_=64, nbytes=None):
        need = lib.ttt_split_saved_bytes(2, 4, 8, K, F_, 0) if nbytes is None else nbytes
        return lib.ttt_linear_fwd(*([P] * 8), 2, 4, 8, K, F_, 4, dtype, rule, 1e-8, P, None, None, None, None, P, need,
                                  None)

    assert fwd(dtype=1) == -2 and fwd(F_=32) == -1 and fwd(K=32) == -1
    need = lib.ttt_split_saved_bytes(2, 4, 8, 16, 64, 0)
    assert need > lib.ttt_linear_saved_bytes(2, 4, 8, 16, 64) and fwd(nbytes=need - 4) == -6
