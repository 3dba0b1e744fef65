"""Workloads of HeadStartLSTM as its users run them, for timing and for comparing outputs.

Each case is one pass through the public module: a training step (forward and backward, with
every parameter gradient), eager or captured with ``GraphedTrainStep``, or a forward without
gradients, in recurrent or in parallel (scan) mode.
"""

import math

import torch

import prlstm_amd
from prlstm_amd.graph import GraphedTrainStep

DEV = torch.device("cuda", 0)
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
EPS = 1e-6  # clamp floor of the scan, the functional's default


def _case(name, mode, call, t, b, d, h, dtype="fp32", hx=False, dx=False):
    """mode: "rec" or "par"; call: "train" (eager step), "graph" (captured step) or "infer" (no
    gradients); hx: initial states given; dx: the input wants a gradient (a layer above another)."""
    c = {"mode": mode, "call": call, "T": t, "B": b, "D": d, "H": h, "dtype": dtype, "hx": hx, "dx": dx}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one step of a stream that carries its state from call to call: the smallest call there is
        _case("rec_stream_step", "rec", "infer", 1, 1, 256, 512, hx=True),
        # scoring a few short sequences with an odd-sized model
        _case("rec_infer_ragged", "rec", "infer", 100, 10, 80, 300),
        # the smallest configured training step
        _case("rec_train_small", "rec", "graph", 32, 16, 64, 128),
        # the headline training step
        _case("rec_train_headline", "rec", "graph", 256, 32, 256, 512),
        # the headline layer at twice the batch
        _case("rec_train_batch64", "rec", "train", 128, 64, 256, 512),
        # an upper layer of a stack in truncated BPTT: a width that is no multiple of a tile, a
        # short window, the state of the window before, and a gradient for the layer below
        _case("rec_train_stacked", "rec", "train", 35, 20, 650, 650, hx=True, dx=True),
        # a half-precision module of middle width
        _case("rec_train_bf16", "rec", "train", 96, 24, 512, 768, dtype="bf16"),
        # the large configured hidden size
        _case("rec_train_large", "rec", "train", 64, 32, 1024, 2048),
        # the configured shape both modes run
        _case("par_train_small", "par", "graph", 128, 32, 256, 256),
        # few channels and a very long sequence, as in signal data
        _case("par_train_narrow", "par", "train", 16384, 2, 64, 256, hx=True, dx=True),
        # a half-precision module on sequences of middle length
        _case("par_train_bf16", "par", "train", 1024, 12, 512, 768, dtype="bf16"),
        # the long-sequence configuration: the largest call
        _case("par_train_long", "par", "train", 4096, 16, 256, 1024),
    ]


def _log_int(rng, lo, hi, odd):
    """An integer spread evenly over the logarithm of [lo, hi]; unless `odd`, of few set bits."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if not odd:
        q = 64 if v >= 256 else 16 if v >= 48 else 4 if v >= 8 else 1
        v = max(q, v // q * q)
    return max(lo, min(hi, v))


def draw(rng):
    mode = rng.choice(["rec", "rec", "rec", "par", "par"])
    call = rng.choice(["train", "train", "graph", "infer"])
    odd = rng.random() < 0.5
    d = _log_int(rng, 16, 1024, odd)
    if mode == "rec":
        t, b, h = _log_int(rng, 1, 256, True), _log_int(rng, 1, 128, odd), _log_int(rng, 32, 2048, odd)
        dtype = rng.choice(["fp32", "fp32", "fp32", "bf16"])
    else:
        t, b, h = _log_int(rng, 64, 16384, True), _log_int(rng, 1, 64, odd), _log_int(rng, 32, 1536, odd)
        dtype = rng.choice(["fp32", "fp32", "bf16", "fp16"])
    c = _case(None, mode, call, t, b, d, h, dtype, hx=rng.random() < 0.4, dx=call == "train" and rng.random() < 0.5)
    top = _case(None, "par", "train", 4096, 16, 256, 1024)
    while work(c)["flops"] > 0.9 * work(top)["flops"] or c["T"] * c["B"] * c["H"] > 0.9 * 4096 * 16 * 1024:
        k = "T" if c["T"] > c["B"] else "B"
        c[k] = max(1, c[k] * 3 // 4)
    return c


def prepare(case, seed):
    t, b, d, h, dt = case["T"], case["B"], case["D"], case["H"], DTYPES[case["dtype"]]
    torch.manual_seed(seed)
    with DEV:
        m = prlstm_amd.HeadStartLSTM(d, h, parallel=case["mode"] == "par")
    g = torch.Generator(device=DEV).manual_seed(seed + 1)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    with torch.no_grad():
        m.a.copy_(0.5 * torch.rand(4, device=DEV, generator=g))  # as training moves it
    m = m.to(dt)
    x = rand(t, b, d).to(dt)
    hx = None
    if case["hx"]:
        # the state a window before would have left: |h| < 1, and c positive (sigmoid g-gate)
        hx = ((0.3 * rand(b, h)).tanh().to(dt), rand(b, h).abs().to(dt))
    state = {"m": m, "x": x, "hx": hx, "call": case["call"], "dx": case["dx"]}
    if case["call"] != "infer":
        state["dout"] = rand(t, b, h).to(dt)
    if case["dx"]:
        x.requires_grad_(True)
    if case["call"] == "graph":
        state["step"] = GraphedTrainStep(m, x, hx=hx, grad_out=state["dout"])
    return state


def _grads(m):
    return {"d" + n: p.grad for n, p in m.named_parameters()}


def run(state):
    m, x, hx = state["m"], state["x"], state["hx"]
    if state["call"] == "infer":
        with torch.no_grad():
            out, (h_n, c_n) = m(x, hx)
        return {"out": out, "h_n": h_n, "c_n": c_n}
    if state["call"] == "graph":
        step = state["step"]
        out = step.step(x)
        return {"out": out, "h_n": step.static_h_n, "c_n": step.static_c_n, **_grads(m)}
    m.zero_grad(set_to_none=True)
    if state["dx"]:
        x.grad = None
    out, (h_n, c_n) = m(x, hx)
    out.backward(state["dout"])
    res = {"out": out.detach(), "h_n": h_n.detach(), "c_n": c_n.detach(), **_grads(m)}
    if state["dx"]:
        res["dx"] = x.grad
    return res


def work(case):
    t, b, d, h = case["T"], case["B"], case["D"], case["H"]
    train, rec = case["call"] != "infer", case["mode"] == "rec"
    w = 4 * h * (d + h + 2) + 4 if rec else 4 * h * (d + 1)  # parameters the mode reads
    n = t * b * (d + h) + w + (4 if case["hx"] else 2) * b * h  # x in, out and states out
    flops = 8 * t * b * h * (d + (h if rec else 0))
    if train:
        n += t * b * h + w + (t * b * d if case["dx"] else 0)  # dout in, gradients out
        flops *= 2
        if rec:
            flops += 8 * t * b * h * h  # dW_hh beside dh
        if case["dx"]:
            flops += 8 * t * b * h * d
    return {"bytes": n * (4 if case["dtype"] == "fp32" else 2), "flops": flops}


def tolerance(case):
    # fp32: every output is within 0.06e-6 to 0.7e-6 of exact() (the gradient of a, a sum with
    # cancellation, is the furthest), so two correct implementations differ by up to 1.4e-6.
    # 16-bit modules round their outputs and gradients: 1.7e-3 from exact() in bf16.
    return {"rel": 5e-6, "max": 5e-4} if case["dtype"] == "fp32" else {"rel": 7e-3, "max": 3e-2}


def exact(case, seed):
    """What run() returns, in 64 bits on plain torch operations."""
    if case["call"] == "graph":
        case = dict(case, call="train")  # the same inputs, without a capture
    s = prepare(case, seed)
    t, b, d, h = case["T"], case["B"], case["D"], case["H"]
    m, rec, train = s["m"], case["mode"] == "rec", case["call"] != "infer"
    with torch.no_grad():
        w_ih, w_hh, b_ih, b_hh, a = (p.double() for p in (m.weight_ih_l0, m.weight_hh_l0, m.bias_ih_l0,
                                                          m.bias_hh_l0, m.a))
        x = s["x"].double().reshape(t * b, d)
        zero = torch.zeros(b, h, dtype=torch.float64, device=DEV)
        h0, c0 = (zero, zero) if s["hx"] is None else (v.double() for v in s["hx"])
        z = (x @ w_ih.t() + b_ih).reshape(t, b, 4, h)
        if rec:
            ag = a.repeat_interleave(h)
            w_s, b_s = ag[:, None] * w_hh, ag * b_hh
            hs = torch.empty(t + 1, b, h, dtype=torch.float64, device=DEV)
            cs = torch.empty_like(hs)
            hs[0], cs[0] = h0, c0
            act = torch.empty_like(z)
            for k in range(t):
                act[k] = torch.sigmoid(z[k] + torch.addmm(b_s, hs[k], w_s.t()).view(b, 4, h))
                cs[k + 1] = act[k][:, 1] * cs[k] + act[k][:, 0] * act[k][:, 2]
                hs[k + 1] = act[k][:, 3] * cs[k + 1].tanh()
            out = hs[1:]
        else:
            act = torch.sigmoid(z)
            f, ig = act[:, :, 1], act[:, :, 0] * act[:, :, 2]
            fc, bc = f.clamp_min(EPS), ig.clamp_min(EPS)
            cs = torch.empty(t + 1, b, h, dtype=torch.float64, device=DEV)
            cs[0] = c0.clamp_min(EPS)
            for k in range(t):
                torch.addcmul(bc[k], fc[k], cs[k], out=cs[k + 1])
            out = act[:, :, 3] * cs[1:].tanh()
        res = {"out": out, "h_n": out[-1][None], "c_n": cs[-1][None]}
        if not train:
            return res
        dout = s["dout"].double()
        i, f, g, o = act.unbind(2)
        tc = cs[1:].tanh()
        dz = torch.empty_like(z)
        if rec:
            dh, dc = zero, zero
            for k in range(t - 1, -1, -1):
                dh = dh + dout[k]
                dc = dc + dh * o[k] * (1 - tc[k] * tc[k])
                dz[k, :, 0] = dc * g[k] * i[k] * (1 - i[k])
                dz[k, :, 1] = dc * cs[k] * f[k] * (1 - f[k])
                dz[k, :, 2] = dc * i[k] * g[k] * (1 - g[k])
                dz[k, :, 3] = dh * tc[k] * o[k] * (1 - o[k])
                dh = dz[k].reshape(b, 4 * h) @ w_s
                dc = dc * f[k]
        else:
            gc = dout * o * (1 - tc * tc)  # becomes the gradient of c_t
            for k in range(t - 2, -1, -1):
                gc[k].addcmul_(fc[k + 1], gc[k + 1])
            gb = gc * (ig >= EPS)
            dz[:, :, 0] = gb * g * i * (1 - i)
            dz[:, :, 1] = gc * cs[:-1] * (f >= EPS) * f * (1 - f)
            dz[:, :, 2] = gb * i * g * (1 - g)
            dz[:, :, 3] = dout * tc * o * (1 - o)
        dz = dz.reshape(t * b, 4 * h)
        db = dz.sum(0)
        res.update(dweight_ih_l0=dz.t() @ x, dweight_hh_l0=None, dbias_ih_l0=db, dbias_hh_l0=None, da=None)
        if rec:
            dw_s = dz.t() @ hs[:-1].reshape(t * b, h)
            res["dweight_hh_l0"] = ag[:, None] * dw_s
            res["dbias_hh_l0"] = ag * db
            res["da"] = ((w_hh * dw_s).sum(1) + b_hh * db).view(4, h).sum(1)
        if s["dx"]:
            res["dx"] = (dz @ w_ih).reshape(t, b, d)
        return res
