"""Performance cases: the work that programs have this framework do, through
its public entry points, over the range of sizes, types and options in use.

A case is a dict of plain values.  ``kind`` says what a pass is:

  forward   inference: O of ``triton_attention`` under ``no_grad``
  train     forward and first backward (dQ, dK, dV), no second order
  step      forward, backward with ``create_graph=True`` and the double
            backward (the vector-Jacobian product of dQ, dK, dV with given
            cotangents): the meta-learning step of the attention
  window    ``step`` through ``windowed_attention`` (no mask tensor)
  masked    ``step`` through ``gradgrad_attention`` with an additive mask,
            square or with fewer queries than keys (a chunk and its history)
  layer     ``WindowedSelfAttention``: output, gradients of its four weights
            with ``create_graph=True``, and their double backward

Backward passes run on the calling thread (as ``bench.py`` does): the default
hand-off to autograd's device thread costs more than the kernels of a small
call.
"""
from __future__ import annotations

import math

import torch

from testtimeideas_amd.ttt_e2e.attention import WindowedSelfAttention, gradgrad_attention, windowed_attention
from testtimeideas_amd.ttt_e2e.utils import local_window_mask
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, b, h, t, d, dtype, *, causal=True, mode="recompute", window=0, local=True, tk=0, mask="",
          qkv_scale=1.0):
    c = dict(kind=kind, b=b, h=h, t=t, tk=tk or t, d=d, dtype=dtype, causal=causal, mode=mode, window=window,
             local=local, mask=mask, qkv_scale=qkv_scale)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one short prompt through a small layer at inference: latency of one call
        _case("forward_t128", "forward", 1, 4, 128, 64, "fp16"),
        # prefill of a batch of ordinary prompts of a 16-head, d = 128 model at inference
        _case("forward_t4096_d128", "forward", 2, 16, 4096, 128, "bf16"),
        # the smallest point of the grad-grad sweep: launches and host work count
        _case("step_t512", "step", 1, 1, 512, 64, "fp16", mode="save_p_triton_full"),
        # the middle of the sweep, without the causal mask
        _case("step_t2048_full", "step", 1, 1, 2048, 64, "fp16", causal=False, mode="save_p_triton_full"),
        # the headline step
        _case("step_t8192", "step", 1, 1, 8192, 64, "fp16", mode="save_p_triton_full"),
        # the largest point of the sweep, in the default mode (P recomputed)
        _case("step_t16384", "step", 1, 1, 16384, 64, "fp16"),
        # first-order training of an eight-head layer, P kept
        _case("train_t2048_d128", "train", 2, 4, 2048, 128, "fp16", causal=False, mode="save_p"),
        # a head dim and a length that fill no tile: first-order training of an 80-wide head
        _case("train_t1000_d80", "train", 2, 8, 1000, 80, "bf16"),
        # the largest step: a 16-head layer at 8k tokens
        _case("step_b4_t8192_d128", "step", 4, 16, 8192, 128, "bf16", mode="save_p_triton_full", qkv_scale=0.5),
        # the test-time-training model's inner-loop chunk: six heads, window 512, fp32, as one layer call
        _case("layer_t1024_fp32", "layer", 8, 6, 1024, 64, "fp32", window=512),
        # the same attention over a whole 8k sequence in bf16
        _case("window_t8192", "window", 8, 6, 8192, 64, "bf16", window=512),
        # a chunk of queries against its longer history, with the model's additive window mask
        _case("masked_t512_k2048", "masked", 2, 6, 512, 64, "fp32", tk=2048, causal=False, mask="window", window=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: lengths over their logarithm (odd
    ones among them), both 16-bit types and fp32, the head dims of the tests."""
    save = ["save_p", "save_p_triton_full"]
    while True:
        kind = rng.choice(["forward", "train", "step", "step", "window", "masked", "layer"])
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        d = rng.choice([64, 64, 128, 128, 32, 80])
        b, h = rng.choice([1, 1, 2, 4, 8]), rng.choice([1, 2, 4, 6, 8, 16])
        if kind in ("forward", "train", "step"):
            c = _case("", kind, b, h, _log_int(rng, 64, 16384), d, dtype, causal=rng.random() < 0.7,
                      mode=rng.choice(save + ["recompute", "recompute"]), qkv_scale=0.5 if d == 128 else 1.0)
        elif kind == "window":
            t = _log_int(rng, 256, 8192)
            c = _case("", kind, b, h, t, d, dtype, window=rng.choice([128, 256, 512]), local=rng.random() < 0.7,
                      mode=rng.choice(save + ["recompute"] * 3))
        elif kind == "masked":
            tk = _log_int(rng, 64, 4096)
            t = tk if rng.random() < 0.5 else max(1, int(tk * rng.uniform(0.1, 0.9)))
            c = _case("", kind, b, h, t, d, dtype, causal=False, tk=tk, mask=rng.choice(["window", "padding"]),
                      window=rng.choice([128, 512, 1024]))
        else:
            c = _case("", kind, rng.choice([1, 2, 4, 8]), rng.choice([4, 6, 8]), _log_int(rng, 128, 4096), 64, "fp32",
                      window=rng.choice([256, 512]))
        # no costlier than the largest listed case: its operations at the types' rates, and its P
        cap = work(listed()[8])["flops"]
        if work(c)["flops"] * (16 if dtype == "fp32" or kind == "layer" else 1) <= cap and \
                c["b"] * c["h"] * c["tk"] ** 2 <= 2 ** 32:
            return c


# ---------------------------------------------------------------------------
# What a program holds before the call.
# ---------------------------------------------------------------------------
def _mask(case, device):
    """The additive mask of a ``masked`` case (fp32, as the model builds it)."""
    t, tk = case["t"], case["tk"]
    if case["mask"] == "window":
        return local_window_mask(tk - t, tk, 0, tk, case["window"], device, torch.float32)
    # key padding: batch entry i holds tk - 37 i keys (at least half of them)
    m = torch.zeros((case["b"], 1, 1, tk), dtype=torch.float32, device=device)
    for i in range(case["b"]):
        m[i, ..., max(tk - 37 * i, (tk + 1) // 2):] = float("-inf")
    return m


def _inputs(case, seed):
    """q, k, v, dO and the cotangents rq, rk, rv of an attention case."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    qs, ks = (case["b"], case["h"], case["t"], case["d"]), (case["b"], case["h"], case["tk"], case["d"])
    out = []
    for shape, mul in ((qs, case["qkv_scale"]), (ks, case["qkv_scale"]), (ks, case["qkv_scale"]), (qs, 1.0),
                       (qs, 1.0), (ks, 1.0), (ks, 1.0)):
        out.append((torch.randn(shape, generator=gen, device=dev, dtype=torch.float32) * mul).to(dt))
    return out


def _layer_inputs(case, seed):
    """x, dy, the layer's weights and biases in ``WindowedSelfAttention``'s
    initialisation range, and the weights' cotangents."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dm = case["h"] * case["d"]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32)

    x, dy = randn(case["b"], case["t"], dm), randn(case["b"], case["t"], dm)
    ws = [(torch.rand((dm, dm), generator=gen, device=dev) * 2 - 1) / math.sqrt(dm) for _ in range(4)]
    bs = [(torch.rand((dm,), generator=gen, device=dev) * 2 - 1) / math.sqrt(dm) for _ in range(4)]
    return x, dy, ws, bs, [randn(dm, dm) for _ in range(4)]


def prepare(case, seed):
    if case["kind"] == "layer":
        x, dy, ws, bs, rs = _layer_inputs(case, seed)
        layer = WindowedSelfAttention(case["h"] * case["d"], case["h"], case["window"]).to("cuda")
        projs = (layer.q_proj, layer.k_proj, layer.v_proj, layer.out_proj)
        with torch.no_grad():
            for p, w, b in zip(projs, ws, bs):
                p.weight.copy_(w)
                p.bias.copy_(b)
        return dict(case=case, layer=layer, weights=[p.weight for p in projs], x=x.requires_grad_(), dy=dy, rs=rs)
    q, k, v, do, rq, rk, rv = _inputs(case, seed)
    if case["kind"] != "forward":
        for t in (q, k, v):
            t.requires_grad_()
    mask = _mask(case, q.device) if case["kind"] == "masked" else None
    return dict(case=case, q=q, k=k, v=v, do=do, r=(rq, rk, rv), mask=mask)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        with torch.no_grad():
            return triton_attention(state["q"], state["k"], state["v"], causal=case["causal"], bwd_mode=case["mode"])
    with torch.autograd.set_multithreading_enabled(False):
        if kind == "layer":
            y = state["layer"](state["x"])
            gw = torch.autograd.grad(y, state["weights"], state["dy"], create_graph=True)
            meta = torch.autograd.grad(gw, state["weights"] + [state["x"]], state["rs"])
            return [y.detach(), *(g.detach() for g in gw), *meta]
        q, k, v = state["q"], state["k"], state["v"]
        if kind == "masked":
            o = gradgrad_attention(q, k, v, state["mask"], bwd_mode=case["mode"])
        elif kind == "window":
            o = windowed_attention(q, k, v, case["window"], local=case["local"], bwd_mode=case["mode"])
        else:
            o = triton_attention(q, k, v, causal=case["causal"], bwd_mode=case["mode"])
        if kind == "train":
            return [o.detach(), *torch.autograd.grad(o, (q, k, v), state["do"])]
        first = torch.autograd.grad(o, (q, k, v), state["do"], create_graph=True)
        second = torch.autograd.grad(first, (q, k, v), state["r"])
        return [o.detach(), *(g.detach() for g in first), *second]


# ---------------------------------------------------------------------------
# The work of a pass, and its result in 64 bits.
# ---------------------------------------------------------------------------
def _window_lo(case, m):
    """First key that query m of a windowed case sees."""
    t, w = case["t"], case["window"]
    if w <= 0 or w >= t:
        return 0
    if not case["local"]:
        return max(0, m - w + 1)
    return max(0, min(t, (m // w + 1) * w) - w)


def _pairs(case):
    """Visible (query, key) pairs of one (b, h) slice."""
    t, tk = case["t"], case["tk"]
    if case["kind"] in ("window", "layer"):
        return sum(m - _window_lo(case, m) + 1 for m in range(t))
    if case["kind"] == "masked":
        if case["mask"] == "window":
            return sum(min(i + 1, case["window"]) for i in range(tk - t, tk))
        return t * sum(max(tk - 37 * i, (tk + 1) // 2) for i in range(case["b"])) // case["b"]
    return t * (t + 1) // 2 if case["causal"] else t * t


def work(case):
    """Each distinct product of the visible pairs once (forward 4, first
    backward 8, double backward 16 times d operations a pair); each input
    read and each output written once.  P is neither."""
    bh, t, tk, d = case["b"] * case["h"], case["t"], case["tk"], case["d"]
    e = 4 if case["dtype"] == "fp32" else 2
    kind = case["kind"]
    products = {"forward": 4, "train": 12}.get(kind, 28)
    flops = float(products * bh * d * _pairs(case))
    if kind == "layer":
        # dO depends on a weight and O's gradient comes back a second time: GdO (4) and another first backward (8);
        # the projections' 4 products, 5 of the first backward, 15 of the double backward
        n, dm = case["b"] * t, case["h"] * d
        flops = float((28 + 12) * bh * d * _pairs(case)) + 24 * 2.0 * n * dm * dm
        return {"bytes": 4.0 * (4 * n * dm + 16 * dm * dm), "flops": flops}
    nq, nk = {"forward": (2, 2), "train": (4, 4)}.get(kind, (6, 8))  # tensors of q's and of k's shape
    byts = float(e * bh * d * (nq * t + nk * tk))
    if kind == "masked":
        byts += 4.0 * (t * tk if case["mask"] == "window" else case["b"] * tk)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """About four times the relative error measured against ``exact``."""
    return {"rel": {"fp16": 2e-3, "bf16": 1.5e-2, "fp32": 8e-6}[case["dtype"]]}


def _hidden(case, device):
    """Boolean [t, tk] of the pairs that a structured mask hides, or None."""
    t = case["t"]
    if case["kind"] == "masked" or not case["causal"]:
        return None
    i = torch.arange(t, device=device)
    hid = i[None, :] > i[:, None]
    if case["kind"] in ("window", "layer"):
        lo = torch.tensor([_window_lo(case, m) for m in range(t)], device=device)
        hid |= i[None, :] < lo[:, None]
    return hid


def _probs(q, k, scale, hidden, add):
    s = torch.matmul(q, k.t()).mul_(scale)
    if hidden is not None:
        s.masked_fill_(hidden, float("-inf"))
    if add is not None:
        s.add_(add)
    return torch.softmax(s, dim=-1)


def _exact_slice(kind, q, k, v, do, gq, gk, gv, scale, hidden, add):
    """Outputs of one (b, h) slice, all operands float64."""
    p = _probs(q, k, scale, hidden, add)
    o = p @ v
    if kind == "forward":
        return [o]
    dp = do @ v.t()
    dp.sub_((dp * p).sum(-1, keepdim=True))  # dP - D
    ds = p * dp
    first = [scale * (ds @ k), scale * (ds.t() @ q), p.t() @ do]
    if kind == "train":
        return [o, *first]
    # cotangents of dS (less its mean under P), of dP, of P (up to a constant of each row) and of the scores
    gds = (gq @ k.t()).add_(q @ gk.t()).mul_(scale)
    gds.sub_((gds * p).sum(-1, keepdim=True))
    gdp = gds * p
    gp = gds.mul_(dp).add_(do @ gv.t())
    gs = gp.sub_((gp * p).sum(-1, keepdim=True)).mul_(p)
    return [o, *first, scale * (ds @ gk + gs @ k), scale * (ds.t() @ gq + gs.t() @ q), gdp.t() @ do]


def _exact_attention(case, xs, add):
    hidden = _hidden(case, xs[0].device)
    scale = 1.0 / math.sqrt(case["d"])
    outs = None
    for b in range(case["b"]):
        for h in range(case["h"]):
            a = None if add is None else (add if add.dim() == 2 else add[b, 0]).double()
            r = _exact_slice(case["kind"], *(x[b, h].double() for x in xs), scale, hidden, a)
            if outs is None:
                outs = [torch.empty((case["b"], case["h"]) + y.shape, dtype=torch.float64, device=y.device) for y in r]
            for y, z in zip(outs, r):
                y[b, h] = z
    return outs


def _exact_layer(case, seed):
    x, dy, ws, bs, rs = (([t.double() for t in y] if isinstance(y, list) else y.double())
                         for y in _layer_inputs(case, seed))
    b, t, h, d = case["b"], case["t"], case["h"], case["d"]
    hidden = _hidden(case, x.device)
    x.requires_grad_()
    for w in ws:
        w.requires_grad_()
    heads = [(x @ w.t() + c).view(b, t, h, d).transpose(1, 2) for w, c in zip(ws[:3], bs[:3])]
    s = (heads[0] @ heads[1].transpose(-1, -2)) / math.sqrt(d)
    o = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1) @ heads[2]
    y = o.transpose(1, 2).reshape(b, t, h * d) @ ws[3].t() + bs[3]
    gw = torch.autograd.grad(y, ws, dy, create_graph=True)
    meta = torch.autograd.grad(gw, [*ws, x], rs)
    return [y.detach(), *(g.detach() for g in gw), *meta]


def exact(case, seed):
    if case["kind"] == "layer":
        # about twenty live matrices of all heads' scores under autograd
        if case["b"] * case["h"] * case["t"] ** 2 * 8 * 20 > 120e9:
            return None
        return _exact_layer(case, seed)
    xs = _inputs(case, seed)
    add = _mask(case, xs[0].device) if case["kind"] == "masked" else None
    out = _exact_attention(case, xs, add)
    return out[0] if case["kind"] == "forward" else out
