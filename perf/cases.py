"""Performance cases of the scans: what a program that trains or serves linear-recurrence
layers has this package do, through its public functions.

Kinds and their ranges (`draw` spreads cases over them; `listed` holds one or two of each):

    ssd_train      ssd_scan forward + backward, one decay rate per head, bf16
    ssd_general    the same with a dense A_neg [H, N], fp32 / fp16 / bf16
    ssd_prefill    ssd_scan_with_state forward from a cached state (a prompt, or its next piece);
                   prompts come at any length, so L is a multiple of 8 only and seg follows it
    ssd_step       one decoded token on a cached state
    gla_train, gla_prefill, gla_step   the same for gated linear attention
    rglru_train    rglru_gated_scan forward + backward (the gate math in the kernels)
    rglru_plain    rglru_scan forward + backward (a and the gated input from outside)
    rotlru_train   rotlru_scan forward + backward
    gdn_train      gated_deltanet_scan forward + backward

Input distributions are those of the benchmark.  A training pass returns y and every gradient.
Passes whose kernels take some tens of microseconds are launch-bound from Python, and programs
that run them in earnest capture them in a HIP graph: those cases ("graph") capture one step of
the public functions in `prepare` and replay it in `run`.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-recurrence_amd"))

import mlx_recurrence_amd as mr  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ITEM = {"f32": 4, "bf16": 2, "f16": 2}
SEG_EXACT = 64   # steps per re-computed segment of exact()


def listed():
    return [
        # decoding one sequence of a wide model: latency, one launch per layer and token
        dict(name="ssd_step_one", kind="ssd_step", dtype="bf16", B=1, H=80, Dh=64, N=128),
        # decoding a full serving batch: the state's read and write
        dict(name="gla_step_batch", kind="gla_step", dtype="bf16", B=64, H=12, Dh=128),
        # one training layer of a small model, inside a captured step
        dict(name="ssd_train_small", kind="ssd_train", dtype="bf16", B=3, L=512, H=12, Dh=64, N=16, seg=32,
             graph=True),
        dict(name="gla_train_small", kind="gla_train", dtype="bf16", B=3, L=512, H=12, Dh=64, seg=32, graph=True),
        # one training layer of a large model: long sequences, wide state
        dict(name="ssd_train_large", kind="ssd_train", dtype="bf16", B=8, L=4096, H=80, Dh=64, N=128, seg=32,
             graph=False),
        # the general contract (decay per head and state, fp32 inputs) at a wide head
        dict(name="ssd_general_f32", kind="ssd_general", dtype="f32", B=3, L=512, H=12, Dh=128, N=64, seg=32,
             graph=False),
        # prompts of a length that is no multiple of 32, continued from a cached state
        dict(name="ssd_prefill_ragged", kind="ssd_prefill", dtype="bf16", B=4, L=1000, H=80, Dh=64, N=128, seg=8),
        # an ordinary training batch of linear attention with wide heads
        dict(name="gla_train_wide", kind="gla_train", dtype="bf16", B=8, L=2048, H=12, Dh=128, seg=32, graph=False),
        # the recurrent layers of a 2560-wide model at a training batch
        dict(name="rglru_train", kind="rglru_train", dtype="bf16", B=8, L=4096, D=2560, seg=32),
        dict(name="rotlru_train", kind="rotlru_train", dtype="bf16", B=8, L=4096, D=2560, seg=32),
        # delta-rule layers: a small captured step and an ordinary training batch
        dict(name="gdn_train_small", kind="gdn_train", dtype="bf16", B=3, L=512, H=12, Dh=64, seg=32, graph=True),
        dict(name="gdn_train", kind="gdn_train", dtype="bf16", B=8, L=2048, H=12, Dh=64, seg=32, graph=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _seg_of(L):
    for s in (32, 16, 8):
        if L % s == 0:
            return s
    raise ValueError(L)


def draw(rng):
    kind = rng.choice(["ssd_train", "ssd_train", "ssd_general", "ssd_prefill", "ssd_step", "gla_train", "gla_train",
                       "gla_prefill", "gla_step", "rglru_train", "rglru_plain", "rotlru_train", "gdn_train"])
    c = dict(kind=kind)
    if kind.endswith("_step"):
        c.update(dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), B=_log_int(rng, 1, 128), H=_log_int(rng, 4, 80),
                 Dh=rng.choice([32, 64, 128]))
        if kind == "ssd_step":
            c["N"] = rng.choice([16, 32, 64, 128])
        return c
    if kind in ("rglru_train", "rglru_plain", "rotlru_train"):
        c.update(dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), L=8 * _log_int(rng, 8, 512))
        c["D"] = (64 if kind == "rotlru_train" else 32) * _log_int(rng, 2, 60)
        c["B"] = max(1, min(_log_int(rng, 1, 16), 80_000_000 // (c["L"] * c["D"])))
        c["seg"] = _seg_of(c["L"])
        return c
    # heads: sizes up to about a sixth of the largest listed case's tokens x heads x state
    c["Dh"] = rng.choice([32, 64, 64, 64, 128])
    if kind.startswith("ssd"):
        c["N"] = rng.choice([16, 32, 64, 128])
    if kind == "gdn_train":
        c["Dh"] = rng.choice([32, 64, 64, 64])
    state = c["Dh"] * c.get("N", c["Dh"])
    c["L"] = 8 * _log_int(rng, 4, 512) if kind.endswith("prefill") else 32 * _log_int(rng, 2, 128)
    c["H"] = _log_int(rng, 1, 80)
    most = max(1, int(3.5e9 / (c["L"] * c["H"] * state)))
    c["B"] = min(_log_int(rng, 1, 16), most)
    c["seg"] = _seg_of(c["L"])
    c["dtype"] = "bf16"
    if kind == "ssd_general":
        c["dtype"] = rng.choice(["f32", "f32", "f16", "bf16"])
        c["N"] = rng.choice([16, 24, 32, 64])
    elif kind in ("gla_train", "gla_prefill") and rng.random() < 0.3:
        c["dtype"] = "f32"
    if not kind.endswith("prefill"):
        c["graph"] = c["B"] * c["L"] * c["H"] <= 40_000
    return c


# ------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """Differentiable inputs (in the functions' argument order), then the upstream gradient or the
    cached state, all on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 1_000_003 + 17)
    dt = DTYPES[case["dtype"]]

    def n(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    def un(*shape):
        return torch.rand(shape, generator=g, device="cuda")

    kind, B = case["kind"], case["B"]
    family = kind.split("_")[0]
    if family in ("rglru", "rotlru"):
        L, D = case["L"], case["D"]
        x, dy = n(B, L, D).to(dt), n(B, L, D)
        if family == "rotlru":
            a = torch.sigmoid(n(B, L, D // 2) + 2.0).to(dt)
            th = (un(B, L, D // 2) * 2 - 1) * math.pi * 0.1
            return [a, torch.cos(th).to(dt), torch.sin(th).to(dt), x], dy
        r, i = n(B, L, D), torch.sigmoid(n(B, L, D))
        base = un(D) * 0.099 + 0.9
        if kind == "rglru_train":
            return [r.to(dt), i.to(dt), x, torch.log(torch.expm1(-torch.log(base)))], dy
        a = base ** (8.0 * torch.sigmoid(r))
        return [a.to(dt), (torch.sqrt(1 - a * a) * i * x).to(dt)], dy
    H, Dh = case["H"], case["Dh"]
    lead = (B, H) if kind.endswith("step") else (B, case["L"], H)
    cols = case["N"] if family == "ssd" else Dh
    if family == "ssd":
        u = n(*lead, Dh).to(dt)
        delta = (n(*lead).abs() * 0.1 + 0.01).to(dt)
        Bm, Cm = n(*lead, cols).to(dt), n(*lead, cols).to(dt)
        A = -torch.exp(un(H, cols) * math.log(16.0)) if kind == "ssd_general" else -torch.exp(un(H) * math.log(16.0))
        ins = [u, delta, Bm, Cm, A]
    elif family == "gla":
        ins = [(n(*lead, Dh) / math.sqrt(Dh)).to(dt) for _ in range(3)] + [torch.sigmoid(n(*lead) + 2.0).to(dt)]
    else:
        q, k = (torch.nn.functional.normalize(n(*lead, Dh), dim=-1).to(dt) for _ in range(2))
        ins = [q, k, n(*lead, Dh).to(dt), torch.exp(-(0.01 + 0.49 * un(*lead))).to(dt), torch.sigmoid(n(*lead)).to(dt)]
    if kind.endswith("step") or kind.endswith("prefill"):
        return ins, n(B, H, Dh, cols)          # the state left by the tokens before
    return ins, n(*lead, Dh)


def _train_fn(case):
    seg = case["seg"]
    return {
        "ssd_train": lambda u, d, b, c, a: mr.ssd_scan(u, d, b, c, a, seg=seg),
        "ssd_general": lambda u, d, b, c, a: mr.ssd_scan(u, d, b, c, a, seg=seg),
        "gla_train": lambda q, k, v, g: mr.gla_scan(q, k, v, g, seg=seg),
        "rglru_train": lambda r, i, x, lam: mr.rglru_gated_scan(r, i, x, lam, 8.0, seg=seg),
        "rglru_plain": lambda a, x: mr.rglru_scan(a, x, seg=seg),
        "rotlru_train": lambda a, c, s, x: mr.rotlru_scan(a, c, s, x, seg=seg),
        "gdn_train": lambda q, k, v, a, b: mr.gated_deltanet_scan(q, k, v, a, b, seg=seg),
    }[case["kind"]]


def _train_pass(fn, ins, dy):
    y = fn(*ins)
    return (y.detach(), *torch.autograd.grad(y, ins, dy))


def _capture(step):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def prepare(case, seed):
    ins, more = _inputs(case, seed)
    if case["kind"].endswith("step") or case["kind"].endswith("prefill"):
        return dict(case=case, ins=ins, state=more)
    for t in ins:
        t.requires_grad_(True)
    st = dict(case=case, ins=ins, dy=more, fn=_train_fn(case))
    if case.get("graph"):
        st["graph"], st["out"] = _capture(lambda: _train_pass(st["fn"], ins, more))
    return st


def run(st):
    case, ins, kind = st["case"], st["ins"], st["case"]["kind"]
    if "graph" in st:
        st["graph"].replay()
        return st["out"]
    with torch.no_grad():
        if kind == "ssd_step":
            return mr.ssd_step(*ins, st["state"]), st["state"]
        if kind == "gla_step":
            return mr.gla_step(*ins, st["state"]), st["state"]
        if kind == "ssd_prefill":
            return mr.ssd_scan_with_state(*ins, seg=case["seg"], initial_state=st["state"])
        if kind == "gla_prefill":
            return mr.gla_scan_with_state(*ins, seg=case["seg"], initial_state=st["state"])
    return _train_pass(st["fn"], ins, st["dy"])


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes: each input read once, each output written once (no checkpoints, no re-reads).  Flops:
    the recurrence itself, per token and state element: 5 forward (decay, input, read-out; 8 with the
    delta rule's erase term) and 14 backward (state again, adjoint, one product per gradient; 22)."""
    kind, B, e = case["kind"], case["B"], ITEM[case["dtype"]]
    family = kind.split("_")[0]
    if family in ("rglru", "rotlru"):
        n = B * case["L"] * case["D"]
        streams = {"rglru_train": 3, "rglru_plain": 2, "rotlru_train": 2.5}[kind]
        return dict(bytes=2 * streams * n * e + 8 * n, flops=n * {"rglru_train": 40, "rglru_plain": 6,
                                                                  "rotlru_train": 14}[kind])
    H, Dh = case["H"], case["Dh"]
    rows = B * H * case.get("L", 1)
    cols = case["N"] if family == "ssd" else Dh
    per_row = {"ssd": Dh + 1 + 2 * cols, "gla": 3 * Dh + 1, "gdn": 3 * Dh + 2}[family]
    state = 4 * B * H * Dh * cols
    params = 4 * H * (cols if kind == "ssd_general" else 1) if family == "ssd" else 0
    fwd, bwd = (8, 22) if family == "gdn" else (5, 14)
    if kind.endswith("step") or kind.endswith("prefill"):
        return dict(bytes=rows * (per_row * e + 4 * Dh) + 2 * state + params, flops=fwd * rows * Dh * cols)
    return dict(bytes=rows * (2 * per_row * e + 8 * Dh) + 2 * params, flops=(fwd + bwd) * rows * Dh * cols)


def tolerance(case):
    """About four times the distance to exact() of the present kernels (for prompts: of their bf16
    hi + lo split of fp32 operands; for 16-bit training: of the gradients' storage rounding)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind.endswith("step"):
        return {"rel": 1e-6, "max": 3e-5}
    if kind.endswith("prefill"):
        return {"rel": 1e-5, "max": 2e-4}
    if dtype == "f32":
        return {"rel": 1e-5, "max": 5e-4}
    return {"rel": 7e-3, "max": 3e-2} if dtype == "bf16" else {"rel": 1e-3, "max": 4e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


def _segment(case, h, xs, ps):
    """Per-step recurrence over one segment: xs [steps, ...] streams, ps parameters."""
    kind = case["kind"]
    family = kind.split("_")[0]
    ys = []
    if family == "rglru":
        if kind == "rglru_train":
            r, i, x = xs
            z = -8.0 * _softplus(ps[0]) * torch.sigmoid(r)
            a, x = torch.exp(z), torch.sqrt(-torch.expm1(2 * z)) * (i * x)
        else:
            a, x = xs
        for a_t, x_t in zip(a.unbind(0), x.unbind(0)):
            h = a_t * h + x_t
            ys.append(h)
    elif family == "rotlru":
        a, cs, sn, x = xs
        x = x.unflatten(-1, (-1, 2))
        rc, rs, xu, xw = (t.unbind(0) for t in (a * cs, a * sn, x[..., 0], x[..., 1]))
        hu, hw = h.unflatten(-1, (-1, 2)).unbind(-1)
        for c_t, s_t, u_t, w_t in zip(rc, rs, xu, xw):
            hu, hw = c_t * hu - s_t * hw + u_t, s_t * hu + c_t * hw + w_t
            ys.append(torch.stack((hu, hw), -1).flatten(-2))
        h = ys[-1]
    elif family == "ssd":
        u, d, b, c = xs
        A = ps[0] if ps[0].ndim == 2 else ps[0][:, None]
        dec = torch.exp(d.unsqueeze(-1) * A)
        for e_t, b_t, c_t, u_t in zip(dec.unbind(0), (d.unsqueeze(-1) * b).unbind(0), c.unbind(0), u.unbind(0)):
            h = e_t[..., None, :] * h + u_t[..., :, None] * b_t[..., None, :]
            ys.append((h * c_t[..., None, :]).sum(-1))
    elif family == "gla":
        for q_t, k_t, v_t, g_t in zip(*(t.unbind(0) for t in xs)):
            h = g_t[..., None, None] * h + k_t[..., :, None] * v_t[..., None, :]
            ys.append((q_t[..., :, None] * h).sum(-2))
    else:
        for q_t, k_t, v_t, a_t, b_t in zip(*(t.unbind(0) for t in xs)):
            w = b_t[..., None] * (v_t - a_t[..., None] * (k_t[..., :, None] * h).sum(-2))
            h = a_t[..., None, None] * h + k_t[..., :, None] * w[..., None, :]
            ys.append((q_t[..., :, None] * h).sum(-2))
    return torch.stack(ys), h


def exact(case, seed):
    ins, more = _inputs(case, seed)
    kind = case["kind"]
    family = kind.split("_")[0]
    params = {"ssd": 1, "rglru": 1 if kind == "rglru_train" else 0}.get(family, 0)
    ins = [t.double() for t in ins]
    xs, ps = ins[:len(ins) - params], ins[len(ins) - params:]
    step = kind.endswith("step")
    xs = [t.unsqueeze(0) if step else t.transpose(0, 1) for t in xs]       # [L, B, ...]
    L = xs[0].shape[0]
    serve = step or kind.endswith("prefill")
    if serve:
        h = more.double()
    elif family in ("rglru", "rotlru"):
        h = torch.zeros(case["B"], case["D"], dtype=torch.float64, device="cuda")
    else:
        h = torch.zeros(case["B"], case["H"], case["Dh"], case["N"] if family == "ssd" else case["Dh"],
                        dtype=torch.float64, device="cuda")
    starts, ys, entering = range(0, L, SEG_EXACT), [], []
    with torch.no_grad():
        for s in starts:
            if not serve:
                entering.append(h)
            y, h = _segment(case, h, [t[s:s + SEG_EXACT] for t in xs], ps)
            ys.append(y)
    y = torch.cat(ys)
    del ys
    if step:
        return y[0], h
    y = y.transpose(0, 1).contiguous()
    if serve:
        return y, h
    dy = more.double().transpose(0, 1)
    grads = [[None] * len(starts) for _ in xs]
    dps = [torch.zeros_like(p) for p in ps]
    dh = torch.zeros_like(h)
    for n in reversed(range(len(starts))):
        s = starts[n]
        leaf = [t.detach().requires_grad_(True) for t in (entering[n], *(t[s:s + SEG_EXACT] for t in xs), *ps)]
        entering[n] = None
        with torch.enable_grad():
            y_s, h_s = _segment(case, leaf[0], leaf[1:1 + len(xs)], leaf[1 + len(xs):])
        got = torch.autograd.grad((y_s, h_s), leaf, (dy[s:s + SEG_EXACT], dh))
        dh = got[0]
        for k in range(len(xs)):
            grads[k][n] = got[1 + k]
        for k in range(len(ps)):
            dps[k] += got[1 + len(xs) + k]
        del y_s, h_s, leaf, got
    return (y, *(torch.cat(g).transpose(0, 1).contiguous() for g in grads), *dps)
