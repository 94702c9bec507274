"""Initial states that a batch shares (expanded from [H,...], TTT_STATE_SHARED) are
read in place: bitwise the outputs and gradients of the same states as a
contiguous [B,H,...], in every kernel family; forms that are not such an
expansion take the contiguous path."""

import pytest
import torch

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


# K, F, FF (0: Linear): the specialised kernels (fp32 Linear: the split form too),
# register-resident, mini-batch in LDS, general
SHAPES = [(16, 64, 0), (16, 32, 0), (16, 64, 256), (16, 32, 128), (16, 64, 64), (64, 32, 32), (64, 32, 0), (64, 64, 64),
          (32, 64, 0), (32, 48, 48), (32, 48, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [F32, BF16, F16])
@pytest.mark.parametrize("K,F_,FF", SHAPES)
def test_bitwise_as_contiguous(K, F_, FF, dt):
    from ttt_amd.linear import TTTLinearFunction
    from ttt_amd.mlp import TTTMLPFunction
    B, H, NC = 3, 2, 3
    x = [torch.nn.functional.normalize(_rand(B, H, NC, K, F_, seed=i), dim=-1).to(dt).cuda() for i in range(3)]
    lr = (0.1 * torch.sigmoid(_rand(B, H, NC, K, seed=4)) / F_).cuda()
    ln = [(1 + 0.1 * _rand(H, F_, seed=5)).cuda(), (0.1 * _rand(H, F_, seed=6)).cuda()]
    shapes = [(H, F_, FF), (H, 1, FF), (H, FF, F_), (H, 1, F_)] if FF else [(H, F_, F_), (H, 1, F_)]
    ps = [0.1 * _rand(*s, seed=7 + i).cuda() for i, s in enumerate(shapes)]
    dout = _rand(B, H, NC, K, F_, seed=12).to(dt).cuda()
    fn = TTTMLPFunction if FF else TTTLinearFunction
    res = []
    for shared in (True, False):
        leaf = [p.clone().requires_grad_(True) for p in ps]
        st = [p.unsqueeze(0).expand(B, -1, -1, -1) for p in leaf]
        if not shared:
            st = [s.contiguous() for s in st]
        out = fn.apply(*ln, *st, *x, lr, 2, *((2,) if FF else ()), 1e-8, "layer")
        outs = list(out) if FF else [out]
        res.append([*outs, *torch.autograd.grad(outs[0], leaf, dout)])
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_which_states_are_shared():
    from ttt_amd._common import states
    p, b = torch.zeros(2, 8, 8), torch.zeros(2, 1, 8)
    ex = lambda t, n=4: t.unsqueeze(0).expand(n, -1, -1, -1)  # noqa: E731
    assert states((ex(p), ex(b)))[1] and states((ex(p), ex(b)))[0][0].data_ptr() == p.data_ptr()
    off = torch.zeros(2 * 64 + 1)[1:].view(2, 8, 8)  # off the 16-byte grid
    for ts in ((ex(p).contiguous(), ex(b)), (ex(p.double()), ex(b)), (ex(p.transpose(1, 2)), ex(b)), (ex(off), ex(b)),
               (p[:1].unsqueeze(1).expand(4, 2, 8, 8), ex(b)), (ex(p, 1), ex(b, 1))):
        got, shared = states(ts)
        assert not shared and all(g.is_contiguous() and g.dtype == torch.float32 and torch.equal(g, t.float())
                                  for g, t in zip(got, ts))
