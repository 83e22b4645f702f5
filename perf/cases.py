"""The work that a user of this framework has it do, as cases to be timed.

Four kinds of case, each through the package's public entry points:

* ``layer``: one training pass of a GRU (``GRU``, ``mse_loss``): forward, loss,
  backward with every gradient, the input's and the initial state's included;
* ``infer``: a forward without autograd (``torch.no_grad``), with carried state;
* ``step``: a whole training step of the benchmark harness's model (GRU stack,
  ``LinearHead``, ``mse_loss``, ``AdamW``);
* ``head``: the head and the loss alone, forward and backward, on a stack's
  output.

``exact`` gives the same results in float64 from plain torch operations.
"""
import math

import torch

from rnn_kernel_amd import GRU, AdamW, LinearHead, mse_loss
from rnn_kernel_amd.harness import BenchmarkModel

DEVICE = "cuda"


def _case(name, kind, L, I, H, B, T, chunks=1, loss="seq", saturate=False, h0=0.1):
    return dict(name=name, kind=kind, L=L, I=I, H=H, B=B, T=T, chunks=chunks, loss=loss, saturate=saturate, h0=h0)


def listed():
    return [
        # the smallest training pass: debugging and unit-test sizes, where
        # launches and the host path are all there is
        _case("small_train", "layer", 1, 16, 16, 2, 8, h0=0.0),
        # online inference, one time step at a time with carried state: the
        # latency of a call through a stack
        _case("online_infer", "infer", 4, 16, 256, 1, 1),
        # the headline workload: one layer, training
        _case("train_h256", "layer", 1, 256, 256, 64, 512),
        # the same layer in inference over whole sequences
        _case("infer_h256", "infer", 1, 256, 256, 64, 512),
        # a hidden size that is no multiple of anything
        _case("train_h129", "layer", 1, 129, 129, 64, 512),
        # a stack on a large batch: the largest training pass
        _case("train_stack", "layer", 2, 256, 256, 256, 1024, h0=0.0),
        # long sequences in chunks with the state carried across, some input
        # rows large enough to saturate the gates
        _case("train_chunked", "layer", 1, 128, 256, 16, 4096, chunks=8, saturate=True, h0=0.5),
        # the harness's model (narrow input, four layers, batch 16) with head,
        # loss and optimiser: a whole training step on a shorter sequence
        _case("harness_step", "step", 4, 16, 256, 16, 2000, h0=0.0),
        # sequence classification on a large batch of short sequences: the
        # loss is on the last state only
        _case("train_last_state", "layer", 1, 64, 128, 400, 128, loss="last", h0=0.0),
        # a wide layer, training
        _case("train_h512", "layer", 1, 512, 512, 64, 256),
        # the widest layer the module takes, inference
        _case("infer_h768", "infer", 1, 768, 768, 32, 256),
        # the head and the loss on a large stack's output
        _case("head_loss", "head", 1, 1, 256, 256, 1024),
    ]


def _flops(case):
    L, I, H, B, T = (case[k] for k in ("L", "I", "H", "B", "T"))
    if case["kind"] == "head":
        return 6.0 * B * T * H
    total = 0.0
    for layer in range(L):
        i = I if layer == 0 else H
        total += 6.0 * B * T * H * (i + H)  # input projection and recurrence
        if case["kind"] != "infer":
            # dh, dW_hh, dW_ih; dx of every layer whose input needs a gradient
            total += 12.0 * B * T * H * H + 6.0 * B * T * H * i
            if layer > 0 or case["kind"] == "layer":
                total += 6.0 * B * T * H * i
    if case["kind"] == "step":
        total += 6.0 * B * T * H
    return total


def _spread(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    # by use: training passes most, then inference, whole steps, the head
    kind = rng.choice(["layer"] * 5 + ["infer"] * 3 + ["step"] + ["head"])
    while True:
        H = _spread(rng, 12, 768)
        B = _spread(rng, 1, 400)
        T = _spread(rng, 1, 2000)
        I = _spread(rng, 1, 768)
        L = rng.choice([1, 1, 2, 3, 4])
        if kind == "head":
            L, I = 1, 1
            if 1 <= B * T <= 256 * 1024:
                break
            continue
        c = dict(kind=kind, L=L, I=I, H=H, B=B, T=T)
        # no more than the listed cases cost: the wide layers' steps weigh more
        if L * T <= 4096 and _flops(c) <= (4e11 if H <= 256 else 1.5e11):
            break
    chunks = rng.choice([1, 1, 1, 4]) if kind == "layer" and T >= 16 else 1
    loss = rng.choice(["seq", "seq", "seq", "last"]) if kind == "layer" and chunks == 1 else "seq"
    h0 = 0.0 if kind == "step" else rng.choice([0.0, 0.1, 0.5])
    c = _case("", kind, L, I, H, B, T, chunks, loss, rng.random() < 0.2, h0)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs ---
def _data(case, seed):
    """Inputs of a case on the GPU: x ~ N(0, 1), with ``saturate`` 5 % of its
    rows ten times larger; h0 ~ N(0, h0^2) (None where it is zero); targets ~
    N(0, 1)."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE)

    L, I, H, B, T = (case[k] for k in ("L", "I", "H", "B", "T"))
    if case["kind"] == "head":
        return torch.tanh(randn(B, T, H)), None, randn(B, T)
    x = randn(B, T, I)
    if case["saturate"]:
        rows = torch.rand(B, T, 1, generator=g, device=DEVICE) < 0.05
        x = torch.where(rows, x * 10.0, x)
    h0 = case["h0"] * randn(L, B, H) if case["h0"] else None
    target = None
    if case["kind"] == "layer":
        target = randn(L, B, H) if case["loss"] == "last" else randn(B, T, H)
    elif case["kind"] == "step":
        target = randn(B, T)
    return x, h0, target


def _module(case, seed):
    torch.manual_seed(seed)  # the modules' own initialisation
    if case["kind"] == "head":
        return LinearHead(case["H"]).to(DEVICE)
    if case["kind"] == "step":
        return BenchmarkModel(case["I"], case["H"], case["L"]).to(DEVICE)
    return GRU(case["I"], case["H"], num_layers=case["L"]).to(DEVICE)


def prepare(case, seed):
    x, h0, target = _data(case, seed)
    model = _module(case, seed)
    if case["kind"] in ("layer", "head"):
        x.requires_grad_(True)
        if h0 is not None:
            h0.requires_grad_(True)
    optimizer = AdamW(model.parameters(), lr=3e-4, weight_decay=1e-4) if case["kind"] == "step" else None
    return dict(case=case, x=x, h0=h0, target=target, model=model, optimizer=optimizer)


# -------------------------------------------------------------------- runs ---
def _grads(model):
    return {name: p.grad for name, p in model.named_parameters()}


def _run_layer(state):
    case, model, x, h0, target = (state[k] for k in ("case", "model", "x", "h0", "target"))
    model.zero_grad(set_to_none=True)
    x.grad = None
    if h0 is not None:
        h0.grad = None
    if case["chunks"] == 1:
        out, hn = model(x, h0)
    else:
        outs, hn = [], h0
        for xc in x.chunk(case["chunks"], dim=1):
            out, hn = model(xc, hn)
            outs.append(out)
        out = torch.cat(outs, dim=1)
    loss = mse_loss(hn if case["loss"] == "last" else out, target)
    loss.backward()
    return dict(loss=loss.detach(), out=out.detach(), hn=hn.detach(), dx=x.grad, dh0=None if h0 is None else h0.grad,
                grads=_grads(model))


def _run_step(state):
    model, optimizer = state["model"], state["optimizer"]
    optimizer.zero_grad(set_to_none=True)
    pred = model(state["x"])
    loss = mse_loss(pred, state["target"])
    loss.backward()
    optimizer.step()
    return dict(loss=loss.detach(), pred=pred.detach(), grads=_grads(model),
                params={name: p.detach() for name, p in model.named_parameters()})


def _run_head(state):
    model, x = state["model"], state["x"]
    model.zero_grad(set_to_none=True)
    x.grad = None
    pred = model(x)
    loss = mse_loss(pred, state["target"])
    loss.backward()
    return dict(loss=loss.detach(), pred=pred.detach(), dx=x.grad, grads=_grads(model))


def run(state):
    kind = state["case"]["kind"]
    if kind == "infer":
        with torch.no_grad():
            out, hn = state["model"](state["x"], state["h0"])
        return dict(out=out, hn=hn)
    return {"layer": _run_layer, "step": _run_step, "head": _run_head}[kind](state)


# -------------------------------------------------------------------- work ---
def work(case):
    L, I, H, B, T = (case[k] for k in ("L", "I", "H", "B", "T"))
    if case["kind"] == "head":
        # the output read once, its gradient written once; targets, predictions
        return dict(bytes=4.0 * (2 * B * T * H + 2 * B * T + 2 * H), flops=_flops(case))
    params = sum(3 * H * ((I if layer == 0 else H) + H + 2) for layer in range(L))
    values = B * T * I + L * B * H + params
    if case["kind"] == "infer":
        values += B * T * H + L * B * H  # the output sequence and the last states
    elif case["kind"] == "layer":
        # output and target (last: one of each per layer), dx, dh0, gradients
        values += B * T * H + (L * B * H if case["loss"] == "last" else B * T * H) + L * B * H
        values += B * T * I + (L * B * H if case["h0"] else 0) + params
    else:
        # targets and predictions; gradients; AdamW reads and writes the
        # parameters and both moments
        values += 2 * B * T + params + 5 * params
    return dict(bytes=4.0 * values, flops=_flops(case))


def tolerance(case):
    # Every value is a float32 sum.  Against exact() the outputs are 1e-7 to
    # 4e-7 off and the gradients 3e-7 to 2e-6 (2-norm), so that two correct
    # orders of summation stay within 1e-5; single small elements of a
    # gradient are off by more of its root mean square.
    if case["kind"] == "step":
        # AdamW divides a gradient by its own size, so that the rounding of
        # the smallest gradients moves their weights
        return dict(rel=1e-4, max=2e-2)
    return dict(rel=1e-5, max=1e-3)


# ------------------------------------------------------------------- exact ---
def _exact_layer(x, h, w_ih, w_hh, b_ih, b_hh):
    """One GRU layer from its equations, in x's data type."""
    H = h.shape[1]
    gx = (x @ w_ih.t() + b_ih).unbind(1)
    w = w_hh.t()
    outs = []
    for g in gx:
        a = torch.addmm(b_hh, h, w)
        rz = torch.sigmoid(g[:, :2 * H] + a[:, :2 * H])
        r, z = rz[:, :H], rz[:, H:]
        n = torch.tanh(g[:, 2 * H:] + r * a[:, 2 * H:])
        h = n + z * (h - n)
        outs.append(h)
    return torch.stack(outs, dim=1), h


def _exact_stack(case, params, prefix, x, h0):
    states = []
    for layer in range(case["L"]):
        w = [params[f"{prefix}{n}_l{layer}"] for n in ("weight_ih", "weight_hh", "bias_ih", "bias_hh")]
        h = h0[layer] if h0 is not None else x.new_zeros(x.shape[0], case["H"])
        x, h = _exact_layer(x, h, *w)
        states.append(h)
    return x, torch.stack(states)


def exact(case, seed):
    x, h0, target = _data(case, seed)
    model = _module(case, seed)
    train = case["kind"] != "infer"
    params = {n: p.detach().double().requires_grad_(train) for n, p in model.named_parameters()}
    x = x.double().requires_grad_(case["kind"] in ("layer", "head"))
    h0 = h0.double().requires_grad_(case["kind"] == "layer") if h0 is not None else None
    target = target.double() if target is not None else None

    def grads():
        return {n: p.grad for n, p in params.items()}

    if case["kind"] == "infer":
        with torch.no_grad():
            out, hn = _exact_stack(case, params, "", x, h0)
        return dict(out=out, hn=hn)
    if case["kind"] == "layer":
        out, hn = _exact_stack(case, params, "", x, h0)
        loss = ((hn if case["loss"] == "last" else out) - target).square().mean()
        loss.backward()
        return dict(loss=loss.detach(), out=out.detach(), hn=hn.detach(), dx=x.grad,
                    dh0=None if h0 is None else h0.grad, grads=grads())
    if case["kind"] == "step":
        out, _ = _exact_stack(case, params, "rnn.", x, None)
        pred = out @ params["head.weight"][0] + params["head.bias"]
        loss = (pred - target).square().mean()
        optimizer = torch.optim.AdamW(params.values(), lr=3e-4, weight_decay=1e-4)
        loss.backward()
        optimizer.step()
        return dict(loss=loss.detach(), pred=pred.detach(), grads=grads(),
                    params={n: p.detach() for n, p in params.items()})
    pred = x @ params["weight"][0] + params["bias"]
    loss = (pred - target).square().mean()
    loss.backward()
    return dict(loss=loss.detach(), pred=pred.detach(), dx=x.grad, grads=grads())
