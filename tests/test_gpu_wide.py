"""The kernels that hold a mini-batch of 32, 48 or 64 tokens in LDS
(csrc/ttt_wide.h) against the CPU oracle at every shape they take, and the
MLP's against the general-shape kernels on the same problem.

Tolerances as for the other kernels: fp32 max-abs <= 1e-4, or 8 times the fp32
oracle's own error against fp64 (tests/_util.fp32_bound); 16 bits rel-L2 <= 2e-2.
The general-shape kernels run the same problem with 16 hidden units more whose
weights and biases are zero: gelu(0) = 0, so these units add exact zeros to
every sum and the two differ by the order of the fp32 sums alone."""

import pytest
import torch

from oracle import ttt_oracle as O
from tests._util import eta_own_dtype, fp32_bound, max_abs, oracle_linear_grads, oracle_mlp_grads, rel_l2, to_dev

pytestmark = pytest.mark.gpu

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
MLP_KEYS = ("ln_w", "ln_b", "W1", "b1", "W2", "b2", "XQ", "XV", "XK", "eta")
LIN_KEYS = ("ln_w", "ln_b", "W1", "b1", "XQ", "XV", "XK", "eta")


def _inputs(B, H, NC, K, F_, FF, dt, kind, seed):
    d = eta_own_dtype(O.make_inputs(B, H, NC, K, F_, FF=FF, seed=seed, dtype=dt, eta_kind=kind, with_grad=True), dt)
    gen = torch.Generator().manual_seed(seed + 1)
    d["ln_w"] = 1 + 0.2 * torch.randn(H, F_, generator=gen)
    d["ln_b"] = 0.2 * torch.randn(H, F_, generator=gen)
    d["b1"] = 0.1 * torch.randn(*d["b1"].shape, generator=gen)
    if FF:
        d["b2"] = 0.1 * torch.randn(*d["b2"].shape, generator=gen)
    return d


def _check(mine, ref, ref32, dt):
    bad = {}
    for k, v in mine.items():
        err, bound = (max_abs(v, ref[k]), fp32_bound(ref[k], ref32[k])) if dt == F32 else (rel_l2(v, ref[k]), 2e-2)
        if not err <= bound:
            bad[k] = (err, bound)
    assert not bad, bad


# one mini-batch, a group that does not divide NC, a group longer than NC
SIZES = [(1, 1, 1, 1, 1), (2, 3, 5, 2, 2), (1, 2, 4, 4, 3)]  # B, H, NC, G, M


@pytest.mark.parametrize("dt,kind", [(F32, "causal"), (BF16, "layer"), (F16, "causal")])
@pytest.mark.parametrize("F_,FF", [(64, 64), (64, 256), (32, 128)])
@pytest.mark.parametrize("K", [32, 48, 64])
def test_mlp(K, F_, FF, dt, kind):
    from ttt_amd.mlp import mlp_backward, mlp_forward
    for B, H, NC, G, M in SIZES[1:] if dt != F32 else SIZES:
        d = _inputs(B, H, NC, K, F_, FF, dt, kind, K + F_ + FF + NC)
        g = to_dev(d)
        out, ck, memo, last, saved = mlp_forward(*(g[k] for k in MLP_KEYS), G, M=M, want_ckpt=True, want_last=True,
                                                 want_saved=True)
        (dlw, dlb, dW1, db1, dW2, db2), (dxq, dxv, dxk, deta) = mlp_backward(
            g["ln_w"], g["ln_b"], g["XQ"], g["XV"], g["XK"], g["eta"], ck, last, saved, g["dOut"], G)
        torch.cuda.synchronize()
        mine = {"out": out}
        for i, nm in enumerate(("W1", "b1", "W2", "b2")):
            mine.update({nm + "_last": last[i], nm + "_ckpt": ck[i], nm + "_memo": memo[i]})
        full = [O.mlp_forward_full(*(d[k].to(t) for k in MLP_KEYS), G=G, M=M) for t in (torch.float64, F32)]
        _check(mine, *full, dt)
        grads = [oracle_mlp_grads(d, d["dOut"], G=0, dtype=t) for t in (torch.float64, F32)]
        _check(dict(dXQ=dxq, dXV=dxv, dXK=dxk, deta=deta, dW1=dW1, db1=db1, dW2=dW2, db2=db2, dln_w=dlw, dln_b=dlb),
               *grads, dt)


@pytest.mark.parametrize("dt,kind", [(F32, "causal"), (BF16, "layer"), (F16, "causal")])
@pytest.mark.parametrize("K", [32, 48, 64])
def test_linear(K, dt, kind):
    from ttt_amd.linear import linear_backward, linear_forward
    for B, H, NC, G, _ in SIZES:
        d = _inputs(B, H, NC, K, 64, 0, dt, kind, K + NC)
        g = to_dev(d)
        out, ck, last, saved = linear_forward(*(g[k] for k in LIN_KEYS), G, want_ckpt=True, want_last=True,
                                              want_saved=True)
        (dlw, dlb, dW1, db1), (dxq, dxv, dxk, deta) = linear_backward(
            g["ln_w"], g["ln_b"], g["XQ"], g["XV"], g["XK"], g["eta"], ck[0], last[0], saved, g["dOut"], G)
        torch.cuda.synchronize()
        full = [O.linear_forward_full(*(d[k].to(t) for k in LIN_KEYS), G=G) for t in (torch.float64, F32)]
        _check({"out": out, "W1_last": last[0], "b1_last": last[1], "W1_ckpt": ck[0], "b1_ckpt": ck[1]}, *full, dt)
        grads = [oracle_linear_grads(d, d["dOut"], G=0, dtype=t) for t in (torch.float64, F32)]
        _check(dict(dXQ=dxq, dXV=dxv, dXK=dxk, deta=deta, dW1=dW1, db1=db1, dln_w=dlw, dln_b=dlb), *grads, dt)


def _pad_units(d, n):
    p = dict(d)
    p["W1"] = torch.nn.functional.pad(d["W1"], (0, n))
    p["b1"] = torch.nn.functional.pad(d["b1"], (0, n))
    p["W2"] = torch.nn.functional.pad(d["W2"], (0, 0, 0, n))
    return p


@pytest.mark.parametrize("rule", ["dense", "dense_f32", "layer", "causal"])
@pytest.mark.parametrize("dt", [F32, BF16, F16])
@pytest.mark.parametrize("K,F_,FF", [(32, 64, 256), (48, 32, 128), (64, 64, 64)])
def test_mlp_matches_the_general_kernels(K, F_, FF, dt, rule):
    """Every eta form and type through the autograd Function, a non-contiguous
    query among the inputs: the same values from both kernel families."""
    from ttt_amd.mlp import TTTMLPFunction
    B, H, NC, n = 2, 2, 3, 16
    d = _inputs(B, H, NC, K, F_, FF, dt, "causal", 5 * K + FF)
    lr = torch.rand(B, H, NC, K, generator=torch.Generator().manual_seed(K)) / F_
    res = []
    for src in (d, _pad_units(d, n)):
        g = to_dev(src)
        g["eta"] = lr.cuda() if rule in ("layer", "causal") else g["eta"].to(F32 if rule == "dense_f32" else dt)
        # (the strides of a [B, NC, K, H, F] tensor)
        g["XQ"] = g["XQ"].permute(0, 2, 3, 1, 4).contiguous().permute(0, 3, 1, 2, 4)
        leaf = {k: g[k].detach().requires_grad_(True) for k in MLP_KEYS}
        out, *memo = TTTMLPFunction.apply(*(leaf[k] for k in MLP_KEYS), 2, 2, O.LN_EPS,
                                          rule if rule in ("layer", "causal") else "dense")
        out.backward(g["dOut"])
        r = {"out": out, **{"d" + k: leaf[k].grad for k in MLP_KEYS}}
        r.update(zip(("W1_memo", "b1_memo", "W2_memo", "b2_memo"), memo))
        res.append(r)
    torch.cuda.synchronize()
    mine, gen = res
    for k in mine:
        a, b = mine[k], gen[k]
        if a.shape != b.shape:  # the padding units
            b = b[tuple(slice(0, s) for s in a.shape)]
        assert a.dtype == b.dtype
        # fp32: sums in another order, through NC = 3 updates; 16-bit outputs:
        # a value at a rounding boundary may round the other way (2^-8, 2^-11),
        # which few do
        tol = 2e-5 if a.dtype == F32 else 2e-3
        if rule == "dense" and dt == F16 and k == "deta":
            assert torch.equal(torch.isfinite(a), torch.isfinite(b))  # past 65504 on these inputs
            a, b = (torch.nan_to_num(t.float(), 0.0, 0.0, 0.0) for t in (a, b))
        assert rel_l2(a, b) <= tol, (k, rel_l2(a, b))
