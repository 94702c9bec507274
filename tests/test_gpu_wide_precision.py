"""The mini-batch-in-LDS kernels' fp32 errors against 64 bits are no larger than those of
the general-shape kernels on the same problem (run with 16 hidden units more whose
weights are zero, see test_gpu_wide.py), the Linear loop's than the fp32 oracle's.

The bound 1.5 on the rms over four inputs is a margin over the spread that two orders of
the same fp32 sums show (0.8 to 1.25 over shapes and inputs); sums that add every term of
an update to the state itself show 2.2 to 2.6."""

import math

import pytest
import torch

from oracle import ttt_oracle as O
from tests._util import oracle_linear_grads, oracle_mlp_grads, rel_l2, to_dev
from tests.test_gpu_wide import LIN_KEYS, MLP_KEYS, _inputs, _pad_units

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
B, H, NC, SEEDS = 1, 2, 8, 4


def _rms(errors):
    return {k: math.sqrt(sum(e[k] ** 2 for e in errors) / len(errors)) for k in errors[0]}


def _run(fn, keys, d, *args):
    g = to_dev(d)
    leaf = {k: g[k].detach().requires_grad_(True) for k in keys}
    out = fn.apply(*(leaf[k] for k in keys), *args)
    out = out[0] if isinstance(out, tuple) else out
    out.backward(g["dOut"])
    return {"out": out.detach(), **{"d" + k: leaf[k].grad for k in ("XQ", "XK", "W1", *(["W2"] if "W2" in keys else []))}}


@pytest.mark.parametrize("K,F_,FF", [(32, 64, 64), (64, 64, 64), (64, 64, 256), (48, 32, 128)])
def test_mlp_against_the_general_kernels(K, F_, FF):
    from ttt_amd.mlp import TTTMLPFunction
    errs = ([], [])
    for seed in range(SEEDS):
        d = _inputs(B, H, NC, K, F_, FF, F32, "layer", 100 * seed + K)
        ref = oracle_mlp_grads(d, d["dOut"], G=0, dtype=F64)
        ref["out"] = O.mlp_forward_full(*(d[k].to(F64) for k in MLP_KEYS), G=2, M=0)["out"]
        for e, src in zip(errs, (d, _pad_units(d, 16))):
            got = _run(TTTMLPFunction, MLP_KEYS, src, 2, 0, O.LN_EPS, "dense")
            e.append({k: rel_l2(v[tuple(slice(0, n) for n in ref[k].shape)].reshape(ref[k].shape), ref[k])
                      for k, v in got.items()})
    mine, gen = map(_rms, errs)
    assert all(mine[k] <= 1.5 * gen[k] for k in mine), (mine, gen)


@pytest.mark.parametrize("K", [32, 64])
def test_linear(K):
    """There is nothing to pad: the fp32 oracle, its sums one matrix product each, is the measure."""
    from ttt_amd.linear import TTTLinearFunction
    errs = ([], [])
    for seed in range(SEEDS):
        d = _inputs(B, H, NC, K, 64, 0, F32, "layer", 100 * seed + K)
        ref, o32 = (oracle_linear_grads(d, d["dOut"], G=0, dtype=t) for t in (F64, F32))
        for r, t in ((ref, F64), (o32, F32)):
            r["out"] = O.linear_forward_full(*(d[k].to(t) for k in LIN_KEYS), G=2)["out"]
        got = _run(TTTLinearFunction, LIN_KEYS, d, 2, O.LN_EPS, "dense")
        for e, src in zip(errs, (got, o32)):
            e.append({k: rel_l2(src[k].cpu().reshape(ref[k].shape), ref[k]) for k in got})
    mine, oracle = map(_rms, errs)
    assert all(mine[k] <= 1.5 * oracle[k] for k in mine), (mine, oracle)
