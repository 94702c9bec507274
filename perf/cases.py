"""The work that users of this framework have it do, as timed and checked cases.

A case is a dict of plain values whose "kind" names the entry point:

  linear      ops.ttt_linear (training or inference) on given XQ, XK, XV, eta
  mlp         TritonMLP.apply, with its memo snapshots where M > 0
  readout     mlp_cached_readout_triton: fixed weights over a sequence
  memo        mlp_memo_combine: the memory-cache combiner over memo states
  layer       TTTWrapper: projections, inner loop, combiner, post-norm, wo
  forecaster  TTTForecaster: input projection, one layer, head

Sizes: B sequences of NC mini-batches of K tokens, H heads of F features, FF
hidden units.  "train" takes the gradient of every input (or parameter) as
well; "dtype" is the activation type (autocast's for layer and forecaster).
"eta" is "causal" (a dense [B,H,NC,K,K] tensor, lr[j]/(i+1) for j <= i, on
inputs drawn from N(0, 1): the benchmark's inner loop) or "layer" (per-token
learning rates that the kernels expand, on L2-normalised queries and keys: what
the layer hands to its inner loop)."""

import contextlib
import math
import os
import sys

import torch
import torch.nn.functional as Fn

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "ttt-triton_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from kernels.mlp_cached_readout import mlp_cached_readout_triton  # noqa: E402
from mlp_triton import TritonMLP  # noqa: E402
from ops.ttt_linear import ttt_linear  # noqa: E402
from ttt_amd.memo import mlp_memo_combine  # noqa: E402
from ttt_amd.model import ModelConfig, TTTForecaster, TTTWrapper  # noqa: E402

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
LN_EPS, READOUT_EPS, POST_EPS = 1e-8, 1e-6, 1e-6
PRED, CHANNELS = 96, 7  # the forecaster's horizon and channels


def listed():
    return [
        # smallest call: one fp32 inference of the Linear op on a short
        # sequence, where launches and one chain's latency are all there is
        dict(name="linear_infer_b2_f32", kind="linear", B=2, H=4, NC=16, K=16, F=64, G=16, dtype="f32", eta="causal",
             train=False),
        # TTT-Linear training at the benchmark's full size
        dict(name="linear_train_b16_bf16", kind="linear", B=16, H=12, NC=128, K=16, F=64, G=16, dtype="bf16",
             eta="causal", train=True),
        # TTT-MLP prefill without gradients, half the benchmark's batch
        dict(name="mlp_infer_b8_bf16", kind="mlp", B=8, H=12, NC=128, K=16, F=64, FF=256, G=8, M=0, dtype="bf16",
             eta="causal", train=False),
        # TTT-MLP training at the benchmark's full size: the headline
        dict(name="mlp_train_b16_bf16", kind="mlp", B=16, H=12, NC=128, K=16, F=64, FF=256, G=8, M=0, dtype="bf16",
             eta="causal", train=True),
        # the same in full precision at odd sizes (5 heads, 37 mini-batches,
        # a checkpoint group that does not divide them)
        dict(name="mlp_train_b3_f32_odd", kind="mlp", B=3, H=5, NC=37, K=16, F=64, FF=256, G=8, M=0, dtype="f32",
             eta="causal", train=True),
        # fixed-weight readout of a whole batch (serving from cached weights)
        dict(name="readout_b16_bf16", kind="readout", B=16, H=12, NC=128, K=16, F=64, FF=256, dtype="bf16"),
        # memory-cache combiner, forward and backward, 16 states per chain
        dict(name="memo_train_b16_bf16", kind="memo", B=16, H=12, NC=128, K=16, F=64, FF=256, M=8, dtype="bf16",
             train=True),
        # the inner loop that the reference's own model configuration runs
        # (K = 64, F = FF = 32, memo every 2 mini-batches), in fp16 as its
        # training script does
        dict(name="mlp_train_k64_f32dim_f16", kind="mlp", B=32, H=4, NC=8, K=64, F=32, FF=32, G=8, M=2, dtype="f16",
             eta="layer", train=True),
        # the same at the default mini-batch of a 256-wide model (4 heads of 64)
        dict(name="mlp_train_k64_f64dim_bf16", kind="mlp", B=32, H=4, NC=8, K=64, F=64, FF=64, G=8, M=2,
             dtype="bf16", eta="layer", train=True),
        # one Linear layer of that model (the configuration's default layer
        # type), training under bf16 autocast
        dict(name="layer_linear_k64_bf16", kind="layer", ssm="ttt_linear", B=32, L=512, D=256, H=4, K=64, M=2,
             dtype="bf16", train=True),
        # a whole forecast of a batch (lookback 512, horizon 96, 7 channels)
        dict(name="forecast_b32_bf16", kind="forecaster", ssm="ttt_mlp", B=32, L=512, D=256, H=4, K=16, M=2,
             dtype="bf16", train=False),
        # the forecaster's training step at the reference's model size in fp32
        dict(name="forecaster_train_b32_f32", kind="forecaster", ssm="ttt_mlp", B=32, L=512, D=128, H=4, K=64, M=2,
             dtype="f32", train=True),
    ]


def draw(rng):
    def span(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["linear", "linear", "mlp", "mlp", "mlp", "readout", "memo", "layer", "forecaster"])
    dt = rng.choice(["bf16", "bf16", "f32", "f16"])
    if kind in ("layer", "forecaster"):
        D, H = rng.choice([(128, 4), (256, 4), (192, 3), (384, 6), (64, 2), (96, 3)])
        K = rng.choice([16, 32, 48, 64])
        c = dict(kind=kind, ssm=rng.choice(["ttt_linear", "ttt_mlp"]), B=span(1, 32), L=K * span(2, max(3, 512 // K)),
                 D=D, H=H, K=K, M=rng.choice([1, 2, 3, 4]), dtype=dt, train=rng.random() < 0.5)
        if c["train"] and c["ssm"] == "ttt_mlp":
            c["dtype"] = "f32"  # in 16 bits the gates' gradients are rounding noise
        return c
    F = rng.choice([32, 64, 64])
    if kind in ("readout", "memo"):
        c = dict(kind=kind, B=span(1, 16), H=span(1, 12), NC=span(4, 128), K=16, F=F, FF=rng.choice([F, 128, 256]),
                 dtype=dt)
        if kind == "memo":
            c.update(M=max(2, c["NC"] // rng.choice([3, 5, 8, 16])), train=rng.random() < 0.5)
        return c
    K = rng.choice([16, 16, 16, 32, 48, 64])
    # the small mini-batches carry the long sequences
    c = dict(kind=kind, B=span(1, 16), H=span(1, 12), NC=span(3, 128 if K == 16 else 512 // K), K=K, F=F,
             G=rng.choice([3, 4, 8, 16]), dtype=dt, eta=rng.choice(["causal", "layer"]), train=rng.random() < 0.6)
    if kind == "mlp":
        c.update(FF=rng.choice([F, 4 * F]), M=rng.choice([0, 0, 2]) if c["NC"] <= 32 else 0)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Draw:
    """Seeded values, made on the GPU (on the CPU in fp32 the same shapes)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * (seed % 4093) + seed)

    def randn(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std


def _inner_inputs(c, r):
    """(XQ, XK, XV, eta or lr, rule) of the inner loop."""
    B, H, NC, K, F, dt = c["B"], c["H"], c["NC"], c["K"], c["F"], DT[c["dtype"]]
    xq, xk, xv = (r.randn(B, H, NC, K, F) for _ in range(3))
    lr = torch.sigmoid(r.randn(B, H, NC, K)) / F
    if c["eta"] == "causal":
        scale = torch.tril(torch.ones(K, K, device="cuda")) / torch.arange(1, K + 1, device="cuda")[:, None]
        eta = lr[..., None, :] * scale
        # in fp16 the dense gradient passes 65504: eta stays in fp32 there
        return xq.to(dt), xk.to(dt), xv.to(dt), eta if dt == torch.float16 else eta.to(dt), "dense"
    xq, xk = Fn.normalize(xq, dim=-1), Fn.normalize(xk, dim=-1)
    d = xv - xk
    xv = (d - d.mean(-1, keepdim=True)) / d.std(-1, keepdim=True) + xk
    return xq.to(dt), xk.to(dt), xv.to(dt), 0.1 * lr, "layer"


def _state(B, H, F, FF, r, mlp):
    """Fast weights of a model: the same for every sequence of the batch."""
    ws = [r.randn(H, F, FF, std=0.02), r.randn(H, 1, FF, std=0.02)]
    if mlp:
        ws += [r.randn(H, FF, F, std=0.02), r.randn(H, 1, F, std=0.02)]
    return [w[None].repeat(B, 1, 1, 1).contiguous() for w in ws]


def _norm_params(H, F, r):
    return 1 + r.randn(H, F, std=0.1), r.randn(H, F, std=0.1)


def _leaves(ts):
    return [t.requires_grad_(True) for t in ts]


def _config(c):
    return ModelConfig(seq_len=c["L"], model_dim=c["D"], num_heads=c["H"], ssm_layer=c["ssm"],
                       mini_batch_size=c["K"], mem_cache_segment_n_mini_batches=c["M"])


def _model(c, seed):
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(seed)
        if c["kind"] == "layer":
            m = TTTWrapper(_config(c))
        else:
            m = TTTForecaster(_config(c), CHANNELS, CHANNELS, PRED)
    return m.cuda()


def prepare(c, seed):
    r = _Draw(seed)
    s = {"c": c, "train": c.get("train", False)}
    kind = c["kind"]
    if kind in ("linear", "mlp"):
        B, H, F = c["B"], c["H"], c["F"]
        xq, xk, xv, eta, s["rule"] = _inner_inputs(c, r)
        ws = _state(B, H, F, c.get("FF", F), r, kind == "mlp")
        s["ln"], s["ws"], s["x"] = list(_norm_params(H, F, r)), ws, [xq, xv, xk, eta]
        if s["train"]:
            s["dout"] = r.randn(B, H, c["NC"], c["K"], F).to(DT[c["dtype"]])
            for part in ("ln", "ws", "x"):
                _leaves(s[part])
    elif kind in ("readout", "memo"):
        B, H, NC, K, F, FF, dt = c["B"], c["H"], c["NC"], c["K"], c["F"], c["FF"], DT[c["dtype"]]
        s["ln"] = list(_norm_params(H, F, r))
        x = [r.randn(B, H, NC, K, F) for _ in range(1 if kind == "readout" else 4)]
        NS = 1 if kind == "readout" else -(-NC // c["M"])
        # weights that have learnt something: pre-activations of order one
        ws = [r.randn(B, H, NS, F, FF, std=F ** -0.5), r.randn(B, H, NS, 1, FF, std=0.1),
              r.randn(B, H, NS, FF, F, std=FF ** -0.5), r.randn(B, H, NS, 1, F, std=0.1)]
        if kind == "readout":
            s["x"], s["ws"] = [x[0].to(dt)], [w[:, :, 0] for w in ws]
        else:
            x[1] = Fn.normalize(x[1], dim=-1)
            s["x"], s["ws"] = [t.to(dt) for t in x], ws
            if s["train"]:
                s["dout"] = r.randn(B, H, NC, K, F).to(dt)
                _leaves(s["x"][1:])
    else:
        s["model"] = _model(c, seed)
        width = c["D"] if kind == "layer" else CHANNELS
        s["x"] = [r.randn(c["B"], c["L"], width)]
        if kind == "layer" and s["train"]:
            s["dout"] = r.randn(c["B"], c["L"], c["D"])
            _leaves(s["x"])
        elif s["train"]:
            s["y"] = r.randn(c["B"], PRED, CHANNELS)
    return s


def _autocast(c):
    dt = DT[c["dtype"]]
    return contextlib.nullcontext() if dt == torch.float32 else torch.autocast("cuda", dtype=dt)


def _trained(model):
    """The parameters that a loss reaches (TTT-Linear never reads XU)."""
    linear = model.config.ssm_layer == "ttt_linear" if hasattr(model, "config") else \
        model.ttt.config.ssm_layer == "ttt_linear"
    return [p for n, p in model.named_parameters() if not (linear and ".wu." in "." + n)]


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    with contextlib.ExitStack() as es:
        if not s["train"]:
            es.enter_context(torch.no_grad())
        return _RUN[s["c"]["kind"]](s, s["c"])


def _run_linear(s, c):
    xq, xv, xk, eta = s["x"]
    if s["rule"] == "dense":
        out = ttt_linear(xk, xq, xv, eta, *s["ln"], *s["ws"], c["G"])  # [B,NC,K,H,F]
        dout = s["dout"].permute(0, 2, 3, 1, 4) if s["train"] else None
    else:
        from linear_triton import TritonLinear
        out = TritonLinear.apply(*s["ln"], *s["ws"], xq, xv, xk, eta, c["G"], LN_EPS, s["rule"])
        dout = s.get("dout")
    if not s["train"]:
        return [out]
    return [out.detach(), *torch.autograd.grad(out, s["x"] + s["ln"] + s["ws"], dout)]


def _run_mlp(s, c):
    xq, xv, xk, eta = s["x"]
    out, *memo = TritonMLP.apply(*s["ln"], *s["ws"], xq, xv, xk, eta, c["G"], c["M"], LN_EPS, s["rule"])
    memo = memo if c["M"] else []
    if not s["train"]:
        return [out, *memo]
    return [out.detach(), *memo, *torch.autograd.grad(out, s["x"] + s["ln"] + s["ws"], s["dout"])]


def _run_readout(s, c):
    return [mlp_cached_readout_triton(s["x"][0], *s["ws"], *s["ln"])]


def _run_memo(s, c):
    xq, xk, xu, xqw = s["x"]
    out = mlp_memo_combine(xq, xk, xu, xqw, *s["ws"], *s["ln"], c["M"])
    if not s["train"]:
        return [out]
    return [out.detach(), *torch.autograd.grad(out, s["x"][1:], s["dout"])]


def _run_layer(s, c):
    with _autocast(c):
        out = s["model"](s["x"][0])
    if not s["train"]:
        return [out]
    return [out.detach(), *torch.autograd.grad(out, s["x"] + _trained(s["model"]), s["dout"].to(out.dtype))]


def _run_forecaster(s, c):
    with _autocast(c):
        pred = s["model"](s["x"][0])
        if not s["train"]:
            return [pred]
        loss = Fn.mse_loss(pred, s["y"])
    return [pred.detach(), loss.detach(), *torch.autograd.grad(loss, _trained(s["model"]))]


_RUN = {"linear": _run_linear, "mlp": _run_mlp, "readout": _run_readout, "memo": _run_memo, "layer": _run_layer,
        "forecaster": _run_forecaster}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _size(c):
    return 4 if c["dtype"] == "f32" else 2


def _inner_work(B, H, NC, K, F, FF, mlp, sx, eta_bytes, train, memo_states=0):
    toks = B * H * NC * K
    flops = toks * (14 * F * FF + 6 * K * FF + 6 * K * F if mlp else 6 * F * F + 6 * K * F)
    state = 4 * ((2 * F * FF + FF + F) if mlp else F * F + F) * B * H
    nbytes = toks * (4 * F * sx + eta_bytes) + state * (1 + memo_states)
    if train:  # dout in; the gradients of the inputs and of the state out
        nbytes += toks * (4 * F * sx + eta_bytes) + state
        flops *= 3
    return nbytes, flops


def work(c):
    kind, sx = c["kind"], _size(c)
    if kind in ("linear", "mlp"):
        e = 4 if c["eta"] == "layer" else c["K"] * (4 if c["dtype"] != "bf16" else 2)
        memo = -(-c["NC"] // c["M"]) if c.get("M") else 0
        b, f = _inner_work(c["B"], c["H"], c["NC"], c["K"], c["F"], c.get("FF", 0), kind == "mlp", sx, e,
                           c["train"], memo)
        return {"bytes": b, "flops": f}
    if kind == "readout":
        toks, st = c["B"] * c["H"] * c["NC"] * c["K"], 4 * (2 * c["F"] * c["FF"] + c["FF"] + c["F"])
        return {"bytes": toks * c["F"] * (sx + 4) + c["B"] * c["H"] * st, "flops": toks * 4 * c["F"] * c["FF"]}
    if kind == "memo":
        NS, T = -(-c["NC"] // c["M"]), c["NC"] * c["K"]
        st = 4 * (2 * c["F"] * c["FF"] + c["FF"] + c["F"])
        pairs = sum(T - (j + 1) * c["M"] * c["K"] for j in range(NS - 1))
        ch = c["B"] * c["H"]
        b, f = ch * (T * c["F"] * 5 * sx + (NS - 1) * st), ch * pairs * 4 * c["F"] * c["FF"]
        # with gradients: dout in, three gradients out; each readout is used twice
        return {"bytes": b + ch * T * c["F"] * 4 * sx * c["train"], "flops": f}
    B, L, D, H, K = c["B"], c["L"], c["D"], c["H"], c["K"]
    mlp, F, NC = c["ssm"] == "ttt_mlp", D // H, L // K
    _, f = _inner_work(B, H, NC, K, F, F, mlp, sx, 4, False)
    out_tokens = B * L if kind == "layer" else B
    f += 2 * B * L * D * (4 * D + H) + 2 * out_tokens * D * D
    params = 5 * D * D + (2 if mlp else 1) * H * F * F
    if mlp and c["M"]:
        NS = -(-NC // c["M"])
        ends = sum(L - (j + 1) * c["M"] * K for j in range(NS - 1))
        f += B * H * ends * 4 * F * F
    if kind == "layer":
        nbytes = 4 * B * L * D * 2 + 4 * params
    else:
        nbytes = 4 * B * (L + PRED) * CHANNELS + 4 * (params + D * PRED * CHANNELS)
        f += 2 * B * L * CHANNELS * D + 2 * B * D * PRED * CHANNELS
    return {"bytes": nbytes * (2 if c["train"] else 1), "flops": f * (3 if c["train"] else 1)}


def tolerance(c):
    """Largest relative differences between correct implementations: about
    four times the outputs' largest errors against 64 bits, as measured (bf16
    7.6e-3, fp16 5e-4 on normalised inputs and a quarter of bf16's on N(0, 1),
    fp32 1e-6 over 37 mini-batches and more over 128; the gates' gradients of
    a layer are differences of nearly equal readouts)."""
    if c["dtype"] == "bf16":
        return {"rel": 2e-2}
    if c["dtype"] == "f16":
        return {"rel": 1e-2}
    return {"rel": 2e-4 if c["kind"] in ("layer", "forecaster") else 2e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _ln(x, w, b, eps):
    d = x - x.mean(-1, keepdim=True)
    return w * (d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps)) + b


def _ln_l2(x, target, w, b, eps):
    """Gradient of |LN(x) - target|^2 / 2 with respect to x."""
    d = x - x.mean(-1, keepdim=True)
    sd = torch.sqrt((d * d).mean(-1, keepdim=True) + eps)
    h = d / sd
    g = (w * h + b - target) * w
    return (g - g.mean(-1, keepdim=True) - h * (g * h).mean(-1, keepdim=True)) / sd


def _gelu(x):
    return Fn.gelu(x, approximate="tanh")


def _dgelu(x):
    k, m = math.sqrt(2 / math.pi), 0.044715
    t = torch.tanh(k * (x + m * x ** 3))
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * k * (1 + 3 * m * x * x)


def _t(x):
    return x.transpose(-1, -2).contiguous()


def _scan(ln, ws, xq, xv, xk, eta, mlp, M=0):
    """(out, memo states): the dual-form recurrence over mini-batches."""
    H, F, NC = xq.shape[1], xq.shape[-1], xq.shape[2]
    w, b = (p.reshape(1, H, 1, F) for p in ln)
    st, outs, memo = list(ws), [], []
    for s in range(NC):
        q, k, v = xq[:, :, s], xk[:, :, s], xv[:, :, s]
        e = eta[:, :, s]
        z1 = k @ st[0] + st[1]
        c1 = e * (q @ _t(k) + 1)
        el = e[:, :, -1:]  # the last row: what reaches the state
        if mlp:
            x2 = _gelu(z1)
            g2 = _ln_l2(x2 @ st[2] + st[3], v - k, w, b, LN_EPS)
            g1 = (g2 @ _t(st[2])) * _dgelu(z1)
            x2b = _gelu(q @ st[0] + st[1] - c1 @ g1)
            z = x2b @ st[2] + st[3] - (e * (x2b @ _t(x2) + 1)) @ g2
            st = [st[0] - (_t(k) * el) @ g1, st[1] - el @ g1, st[2] - (_t(x2) * el) @ g2, st[3] - el @ g2]
        else:
            g1 = _ln_l2(z1, v - k, w, b, LN_EPS)
            z = q @ st[0] + st[1] - c1 @ g1
            st = [st[0] - (_t(k) * el) @ g1, st[1] - el @ g1]
        outs.append(q + _ln(z, w, b, LN_EPS))
        if M and s % M == 0:
            memo.append([p.detach() for p in st])
    memo = [torch.stack(p, 2) for p in zip(*memo)] if M else []
    return torch.stack(outs, 2), memo


def _readout(x, ws, w, b):
    return x + _ln(_gelu(x @ ws[0] + ws[1]) @ ws[2] + ws[3], w, b, READOUT_EPS)


def _combine(xq, xk, xu, xqw, memo, ln, M):
    B, H, NC, K, F = xq.shape
    w, b = (p.detach().reshape(1, H, 1, F) for p in ln)
    seg = [slice(i, min(i + M, NC)) for i in range(0, NC, M)]
    flat = lambda t: t.reshape(B, H, -1, F)  # noqa: E731
    means = [flat(xk[:, :, a]).mean(2) for a in seg]
    outs = [flat(xqw[:, :, seg[0]])]
    for i in range(1, len(seg)):
        q, u = flat(xq[:, :, seg[i]]).detach(), flat(xu[:, :, seg[i]])
        keys = torch.stack([m.detach() for m in means[:i]] + [means[i]], -1)
        gate = torch.softmax(u @ keys, -1)
        o = gate[..., i:] * flat(xqw[:, :, seg[i]])
        for j in range(i):
            o = o + gate[..., j:j + 1] * _readout(q, [p[:, :, j].detach() for p in memo], w, b)
        outs.append(o)
    return torch.cat(outs, 2).reshape(B, H, NC, K, F)


def _rope64(F, L):
    """The rotary table of a one-dimensional sequence (height = width = 1):
    the first F/8 feature pairs turn with the position, the others stay."""
    d = F // 4
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, device="cuda").double() / d))
    ang = torch.zeros(L, F // 2, dtype=torch.float64, device="cuda")
    ang[:, : inv.numel()] = torch.arange(L, device="cuda").double()[:, None] * inv
    return ang


def _rotate(x, ang):
    c, s = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _layer64(c, p, x):
    B, L, D = x.shape
    H, K = c["H"], c["K"]
    F, NC = D // H, L // K
    q, k, v, u = (Fn.linear(x, p[n + ".weight"], p[n + ".bias"]).view(B, L, H, F) for n in ("wq", "wk", "wv", "wu"))
    ang = _rope64(F, L)
    q, k, u = (_rotate(Fn.normalize(t, dim=-1), ang) for t in (q, k, u))
    ln = [p["ttt_norm_weight"], p["ttt_norm_bias"]]
    d = v - k
    v = ln[0] * ((d - d.mean(-1, keepdim=True)) / (d.std(-1, keepdim=True) + 1e-8)) + ln[1] + k
    lr = torch.sigmoid(x @ p["learnable_ttt_lr_weight"][:, 0].t() + p["learnable_ttt_lr_bias"].view(H)) * 0.1 / F
    q, k, v, u = (t.transpose(1, 2).reshape(B, H, NC, K, F) for t in (q, k, v, u))
    lr = lr.transpose(1, 2).reshape(B, H, NC, 1, K)
    eta = (lr / K).expand(B, H, NC, K, K)
    mlp = c["ssm"] == "ttt_mlp"
    ws = [p[n][None].expand(B, -1, -1, -1) for n in (("W1", "b1", "W2", "b2") if mlp else ("W1", "b1"))]
    M = c["M"] if mlp else 0
    out, memo = _scan(ln, ws, q, v, k, eta, mlp, M)
    if M and NC > M:
        out = _combine(q, k, u, out, memo, ln, M)
    h = out.permute(0, 2, 3, 1, 4).reshape(B, L, D)
    h = Fn.layer_norm(h, (D,), p["post_norm.weight"], p["post_norm.bias"], POST_EPS)
    return Fn.linear(h, p["wo.weight"], p["wo.bias"])


def exact(c, seed):
    s = prepare(c, seed)
    kind, train = c["kind"], s["train"]
    up = lambda ts: [t.detach().double().requires_grad_(train) for t in ts]  # noqa: E731
    with contextlib.ExitStack() as es:
        if not train:
            es.enter_context(torch.no_grad())
        if kind in ("linear", "mlp"):
            x, ln, ws = up(s["x"]), up(s["ln"]), up(s["ws"])
            xq, xv, xk, eta = x
            K = c["K"]
            e = (eta / K)[..., None, :].expand(*eta.shape, K) if s["rule"] == "layer" else eta
            out, memo = _scan(ln, ws, xq, xv, xk, e, kind == "mlp", c.get("M", 0))
            dout, ins = s.get("dout"), x + ln + ws
            shown = out.permute(0, 2, 3, 1, 4) if kind == "linear" and s["rule"] == "dense" else out
            first = [shown.detach(), *memo]
        elif kind == "readout":
            ln = [p.double().reshape(1, c["H"], 1, c["F"]) for p in s["ln"]]
            x = s["x"][0].double()
            out = _readout(x.flatten(2, 3), up(s["ws"]), *ln).reshape(x.shape)
            return [out]
        elif kind == "memo":
            x = up(s["x"])
            out = _combine(*x, up(s["ws"]), up(s["ln"]), c["M"])
            dout, ins, first = s.get("dout"), x[1:], [out.detach()]
        else:
            x = up(s["x"])
            named = {n: t for (n, _), t in zip(s["model"].named_parameters(),
                                               up([p for _, p in s["model"].named_parameters()]))}
            mine = {id(p): named[n] for n, p in s["model"].named_parameters()}
            params = [mine[id(p)] for p in _trained(s["model"])]
            if kind == "layer":
                sub = {n[len("ttt."):]: t for n, t in named.items()}
                out = _layer64(c, sub, x[0])
                dout, ins, first = s.get("dout"), x + params, [out.detach()]
                if train and c["dtype"] != "f32":
                    dout = dout.to(DT[c["dtype"]])
            else:
                sub = {n[len("ttt.ttt."):]: t for n, t in named.items() if n.startswith("ttt.ttt.")}
                h = _layer64(c, sub, Fn.linear(x[0], named["in_proj.weight"], named["in_proj.bias"]))
                pred = Fn.linear(h[:, -1], named["head.weight"], named["head.bias"]).view(-1, PRED, CHANNELS)
                if not train:
                    return [pred]
                out = Fn.mse_loss(pred, s["y"].double())
                dout, ins, first = None, params, [pred.detach(), out.detach()]
        if not train:
            return first
        return [*first, *torch.autograd.grad(out, ins, None if dout is None else dout.double())]
