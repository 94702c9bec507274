"""The memory-cache combiner with the readouts' rows kept for its backward
(ttt_mlp_memo_combine_keep / _bwd_kept) against the calls that form the readouts
twice: bitwise the same output and gradients, with and without the memo-state
images; and the bound past which the rows are not kept."""

import pytest
import torch

from tests.test_gpu_memo import GRADS, KEYS, _inputs

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [F32, BF16, F16])
@pytest.mark.parametrize("B,H,NC,F_,FF,M", [
    (2, 2, 7, 64, 64, 2),    # a ragged last segment
    (1, 3, 37, 64, 256, 2),  # 19 states, several chunks
    (2, 2, 19, 32, 128, 3),
    (1, 2, 9, 64, 256, 1),   # one mini-batch per segment
    (1, 2, 2, 32, 32, 1),    # one state, one tile
    (3, 1, 9, 64, 64, 8),    # a single tile past the first segment
])
def test_kept_rows(B, H, NC, F_, FF, M, dt):
    from ttt_amd.memo import (memo_combine_backward, memo_combine_backward_kept, memo_combine_forward, memo_rows,
                              mlp_memo_combine)
    d = {k: v.cuda() for k, v in _inputs(B, H, NC, F_, FF, M, seed=NC + M, dtype=dt).items()}
    args = [d[k] for k in KEYS]
    xq, xk, xu, xqw, *ws, lw, lb = args
    n = memo_rows(B, H, NC, 16, F_, M)
    NS = -(-NC // M)
    assert n == B * H * sum(NC - (j + 1) * M for j in range(NS - 1)) * 16 * (F_ + 1) > 0
    rows = torch.empty(n, device="cuda")
    out0, gates0 = memo_combine_forward(*args, M)
    ref = memo_combine_backward(xq, xu, xqw, *ws, lw, lb, M, gates0, d["dOut"])
    for images in (False, True):
        out, gates = memo_combine_forward(*args, M, images=images, rows=rows)
        assert torch.equal(out, out0)
        got = memo_combine_backward_kept(xq, xu, xqw, lw, lb, M, gates, rows, d["dOut"])
        for a, b in zip(got, ref):
            assert torch.equal(a, b)
    # the autograd function keeps the rows
    leaf = {k: d[k].detach().clone().requires_grad_(k in GRADS) for k in KEYS}
    out = mlp_memo_combine(*(leaf[k] for k in KEYS), M)
    grads = torch.autograd.grad(out, [leaf[k] for k in GRADS], d["dOut"])
    for a, b in zip(grads, got):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_past_the_bound(monkeypatch):
    from ttt_amd import memo
    d = {k: v.cuda() for k, v in _inputs(2, 2, 7, 64, 64, 2, seed=1, dtype=BF16).items()}
    res = []
    for bound in (memo.ROWS_MAX_BYTES, 0):
        monkeypatch.setattr(memo, "ROWS_MAX_BYTES", bound)
        leaf = {k: d[k].detach().clone().requires_grad_(k in GRADS) for k in KEYS}
        out = memo.mlp_memo_combine(*(leaf[k] for k in KEYS), 2)
        assert len(out.grad_fn.saved_tensors) == (7 if bound else 10)
        res.append((out.detach(), *torch.autograd.grad(out, [leaf[k] for k in GRADS], d["dOut"])))
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,NC,F_,FF,M,kept", [
    (4, 8, 61, 64, 64, 4, 10),   # 16 bits, rows past the caches: not kept below 128 hidden units
    (4, 8, 61, 32, 128, 4, 7),   # kept from there on, with the images
])
def test_the_form_that_training_takes(B, H, NC, F_, FF, M, kept):
    from ttt_amd import memo
    d = {k: v.cuda() for k, v in _inputs(B, H, NC, F_, FF, M, seed=3, dtype=BF16).items()}
    leaf = {k: d[k].detach().clone().requires_grad_(k in GRADS) for k in KEYS}
    out = memo.mlp_memo_combine(*(leaf[k] for k in KEYS), M)
    assert len(out.grad_fn.saved_tensors) == kept
    grads = torch.autograd.grad(out, [leaf[k] for k in GRADS], d["dOut"])
    out0, gates0 = memo.memo_combine_forward(*(d[k] for k in KEYS), M, images=False)
    xq, xk, xu, xqw, *ws, lw, lb = (d[k] for k in KEYS)
    ref = memo.memo_combine_backward(xq, xu, xqw, *ws, lw, lb, M, gates0, d["dOut"])
    for a, b in zip((out, *grads), (out0, *ref)):
        assert torch.equal(a, b)


def test_training_form():
    """16 bits keep the rows from 128 hidden units on or where the caches hold
    them, fp32 always; the images are written unless cached rows are kept."""
    from ttt_amd.memo import ROWS_CACHED_BYTES, training_form
    cached, past = ROWS_CACHED_BYTES // 4, ROWS_CACHED_BYTES // 4 + 1
    for dt in (F32, BF16, F16):
        for FF in (32, 64, 128, 256):
            assert training_form(0, FF, dt) == (False, True)
            assert training_form(cached, FF, dt) == (True, False)
            assert training_form(past, FF, dt) == (dt == F32 or FF >= 128, True)


def test_rows_bytes_and_validation():
    from ttt_amd import _lib, memo
    lib = _lib.load()
    assert lib.ttt_mlp_memo_rows_bytes(2, 3, 5, 64, 64, 2) == 2 * 3 * (3 + 1) * 64 * 65 * 4
    assert lib.ttt_mlp_memo_rows_bytes(2, 3, 5, 16, 64, 5) == 0 == lib.ttt_mlp_memo_rows_bytes(2, 3, 5, 16, 64, 9)
    assert lib.ttt_mlp_memo_rows_bytes(2, 3, 5, 16, 48, 2) == 0
    assert memo.memo_rows(16, 12, 128, 16, 64, 8) > 0 and memo.memo_rows(16, 12, 128, 16, 64, 1) == 0  # 0.8 and 6 GB
    P, gb, rb = 0x10000, lib.ttt_mlp_memo_gates_bytes(2, 3, 5, 16, 64, 2), lib.ttt_mlp_memo_rows_bytes(2, 3, 5, 16, 64, 2)
    fwd = lambda rows, n: lib.ttt_mlp_memo_combine_keep(*([P] * 10), 2, 3, 5, 16, 64, 64, 2, 1, 1e-6, P, P, gb, rows,  # noqa: E731
                                                        n, None)
    assert fwd(None, rb) == -3 and fwd(P + 8, rb) == -4 and fwd(P, rb - 4) == -6
    bwd = lambda rows, n, F_=64: lib.ttt_mlp_memo_combine_bwd_kept(*([P] * 6), 2, 3, 5, 16, F_, 2, 1, P, gb, rows, n,  # noqa: E731
                                                                   P, P, P, None)
    assert bwd(None, rb) == -3 and bwd(P, rb - 4) == -6 and bwd(P, rb, 48) == -1
