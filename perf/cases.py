"""The work that users of naju_amd have it do, as cases that can be timed and
checked: the scan itself (streaming decode, prefill, training; state sizes 1
to 128; float32, bfloat16 and float16), the residual block around it, the
training loss, and a training pass of the language model. Every case goes
through a public entry point: naju_amd.naju_scan_hip,
naju_amd.mixer.NajuBlock / NajuLM, naju_amd.xent.cross_entropy.

``listed()`` gives the cases, ``draw(rng)`` further ones of the same ranges,
``prepare`` / ``run`` one of them, ``work`` its unavoidable bytes and flops,
``tolerance`` how far another correct implementation may be off, and
``exact`` what ``run`` returns in float64, in plain torch.
"""
import math

import torch

from naju_amd import naju_scan_hip
from naju_amd.mixer import NajuBlock, NajuLM
from naju_amd.xent import cross_entropy

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}

# the scan's inputs as they are made: forget and input logits N(mean, std).
#   bench: the recipe of the scan benchmark (retention around sigmoid(2))
#   mixer: a mixer at initialisation (gate biases +5 and -2)
#   long:  retention near one (long memories)
#   edge:  10% of the forget gates exactly 0 and 10% exactly 1 (resets)
_GATES = {"bench": (2.0, 1.0, -1.0), "mixer": (5.0, 0.5, -2.0), "long": (4.0, 1.0, 0.0), "edge": (0.0, 2.0, 0.0)}


def _scan(name, mode, batch, time, width, state, dtype, gates_f32=False, h0=False, gates="bench"):
    c = {"kind": "scan", "mode": mode, "batch": batch, "time": time, "width": width, "state": state, "dtype": dtype,
         "gates_f32": gates_f32, "h0": h0, "gates": gates}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one token of streaming decode for 8 sequences of the LM's layer: the state comes in and goes out
        _scan("decode_step", "stream", 8, 1, 1536, 64, "bf16", gates_f32=True, h0=True, gates="mixer"),
        # a small training step: fits the caches, launches and short grids count
        _scan("train_small_f32", "train", 2, 1024, 256, 64, "f32"),
        # the headline workload: the plain gated recurrence (state size 1) with an initial state
        _scan("train_n1_bf16", "train", 8, 4096, 1024, 1, "bf16", h0=True),
        # a long sequence in float32, batch 1: parallel over time only through the chunks
        _scan("train_n1_long_f32", "train", 1, 131072, 2048, 1, "f32", gates="long"),
        # the scan benchmark's first shape at its default type
        _scan("train_f32", "train", 8, 2048, 512, 64, "f32"),
        # the headline shape at the mixer's state size
        _scan("train_bf16", "train", 8, 4096, 1024, 64, "bf16", h0=True),
        # prefill: the forward alone over a long prompt batch
        _scan("prefill_bf16", "infer", 8, 8192, 512, 64, "bf16"),
        # odd sizes, float16, the small state size of a light model
        _scan("train_ragged_f16", "train", 3, 1021, 771, 16, "f16", h0=True),
        # the largest state size
        _scan("train_n128_bf16", "train", 4, 2048, 1024, 128, "bf16"),
        # one residual block (norm, projections, convolutions, scan, readout) of the LM, bf16 autocast
        {"name": "block_train", "kind": "block", "mode": "train", "batch": 8, "time": 2048, "width": 768, "state": 64},
        # the training loss over the LM's vocabulary
        {"name": "loss_train", "kind": "loss", "rows": 16384, "classes": 50257},
        # forward, loss and backward of a language model of four such blocks
        {"name": "lm_train", "kind": "lm", "batch": 8, "time": 2048, "width": 768, "state": 64, "layers": 4,
         "vocab": 50257},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["scan", "block", "loss", "lm"], [8, 2, 1, 1])[0]
    if kind == "scan":
        mode = rng.choices(["train", "infer", "stream"], [5, 2, 1])[0]
        dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
        state = rng.choice([1, 1, 8, 16, 24, 32, 48, 64, 64, 64, 128])
        # widths of real models are multiples of 64; a few are not
        width = 64 * _log(rng, 2, 40) if rng.random() < 0.75 else _log(rng, 100, 2500)
        batch = rng.randint(1, 16)
        time = _log(rng, 1, 64) if mode == "stream" else _log(rng, 128, 16384)
        # as much as the headline shape at most
        time = max(1, min(time, (8 * 4096 * 1024) // (batch * width)))
        return _scan(None, mode, batch, time, width, state, dtype,
                     gates_f32=dtype != "f32" and rng.random() < 0.4, h0=mode == "stream" or rng.random() < 0.3,
                     gates=rng.choice(["bench", "mixer", "long", "edge"]))
    if kind == "loss":
        return {"kind": "loss", "rows": _log(rng, 512, 16384), "classes": _log(rng, 2000, 50257)}
    width, state = rng.choice([256, 320, 512, 768]), rng.choice([16, 32, 64])
    batch = rng.randint(1, 8)
    time = _log(rng, 128, 2048)
    if kind == "block":
        return {"kind": "block", "mode": rng.choice(["train", "train", "infer"]), "batch": batch, "time": time,
                "width": width, "state": state}
    return {"kind": "lm", "batch": batch, "time": time, "width": width, "state": state, "layers": rng.randint(1, 3),
            "vocab": _log(rng, 4000, 50257)}


def _rand(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).add_(mean)


def _scan_inputs(case, seed):
    b, t, d, n = case["batch"], case["time"], case["width"], case["state"]
    dt = _DTYPES[case["dtype"]]
    gt = torch.float32 if case["gates_f32"] else dt
    g = torch.Generator(device="cuda").manual_seed(seed)
    f_mean, f_std, i_mean = _GATES[case["gates"]]
    u = _rand(g, b, t, d).to(dt)
    f = _rand(g, b, t, d, mean=f_mean, std=f_std)
    if case["gates"] == "edge":
        at = torch.rand(b, t, d, generator=g, device="cuda")
        f.masked_fill_(at < 0.1, -math.inf).masked_fill_(at >= 0.9, math.inf)
    f = f.to(gt)
    i = _rand(g, b, t, d, mean=i_mean).to(gt)
    if n == 1:
        bm, cm = torch.ones(b, t, 1, device="cuda", dtype=dt), torch.ones(b, t, 1, device="cuda", dtype=dt)
    else:
        bm, cm = (_rand(g, b, t, n, std=n ** -0.5).to(dt) for _ in range(2))
    skip = _rand(g, d, std=0.01)
    h0 = _rand(g, b, d, n, std=0.1) if case["h0"] else None
    dy = _rand(g, b, t, d).to(dt) if case["mode"] == "train" else None
    return [u, f, i, bm, cm, skip, h0], dy


_SCAN_GRADS = ("du", "df_logit", "di_logit", "dB", "dC", "dD_skip", "dh0")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "scan":
        ins, dy = _scan_inputs(case, seed)
        if case["mode"] == "train":
            for x in ins:
                if x is not None:
                    x.requires_grad_(True)
        return {"case": case, "ins": ins, "dy": dy}
    g = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "loss":
        # logits of a head whose rows are padded to a multiple of 128, as NajuLM's are
        rows, v = case["rows"], case["classes"]
        buf = torch.zeros(rows, -(-v // 128) * 128, device="cuda", dtype=torch.bfloat16)
        buf[:, :v] = torch.randn(rows, v, generator=g, device="cuda", dtype=torch.bfloat16)
        target = torch.randint(0, v, (rows,), generator=g, device="cuda")
        return {"case": case, "logits": buf[:, :v].detach().requires_grad_(True), "target": target}
    torch.manual_seed(seed)
    with torch.device("cuda"):
        if kind == "block":
            model = NajuBlock(case["width"], dropout=0.0, d_state=case["state"], scan_backend="hip")
        else:
            model = NajuLM(case["vocab"], d_model=case["width"], n_layers=case["layers"], dropout=0.0,
                           d_state=case["state"], scan_backend="hip")
    b, t = case["batch"], case["time"]
    if kind == "block":
        x, dy = (_rand(g, b, t, case["width"]) for _ in range(2))
        return {"case": case, "model": model, "x": x.requires_grad_(case["mode"] == "train"), "dy": dy}
    ids = torch.randint(0, case["vocab"], (b, t + 1), generator=g, device="cuda")
    return {"case": case, "model": model, "x": ids[:, :-1].contiguous(), "y": ids[:, 1:].contiguous()}


def _take_grads(params):
    out = {}
    for name, p in params:
        out["d_" + name] = p.grad
        p.grad = None
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "scan":
        ins = state["ins"]
        if case["mode"] == "train":
            y = naju_scan_hip(*ins)
            y.backward(state["dy"])
            out = {"y": y.detach()}
            for name, x in zip(_SCAN_GRADS, ins):
                if x is not None:
                    out[name] = x.grad
                    x.grad = None
            return out
        with torch.no_grad():
            if case["mode"] == "stream":
                y, last = naju_scan_hip(*ins, return_final_state=True)
                return {"y": y, "last": last}
            return {"y": naju_scan_hip(*ins)}
    if kind == "loss":
        logits = state["logits"]
        loss = cross_entropy(logits, state["target"])
        # the head's backward takes the gradient as it comes (no leaf that it would be copied into)
        return {"loss": loss.detach(), "dlogits": torch.autograd.grad(loss, logits)[0]}
    model = state["model"]
    if kind == "block":
        x = state["x"]
        if case["mode"] == "infer":
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
                return {"y": model(x)}
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = model(x)
        y.backward(state["dy"])
        out = {"y": y.detach(), "dx": x.grad, **_take_grads(model.named_parameters())}
        x.grad = None
        return out
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = model(state["x"])
        loss = cross_entropy(logits.view(-1, case["vocab"]), state["y"].view(-1))
    loss.backward()
    return {"logits": logits.detach(), "loss": loss.detach(), **_take_grads(model.named_parameters())}


def _block_work(case):
    """flops of a forward, bytes of its weights (float32)."""
    rows, d, n = case["batch"] * case["time"], case["width"], case["state"]
    di = 2 * d
    weights = 3 * d * di + 2 * di * di + 2 * di * n
    return 2.0 * rows * weights + 5.0 * rows * di * n, 4.0 * weights


def work(case):
    kind = case["kind"]
    if kind == "loss":
        e = case["rows"] * case["classes"]
        return {"bytes": 4.0 * e, "flops": 4.0 * e}
    if kind == "scan":
        b, t, d, n = case["batch"], case["time"], case["width"], case["state"]
        s = 4 if case["dtype"] == "f32" else 2
        sg = 4 if case["gates_f32"] else s
        e, bc, st = b * t * d, b * t * n, 4 * b * d * n
        h0 = st if case["h0"] else 0
        nbytes = e * (2 * s + 2 * sg) + 2 * bc * s + h0 + (st if case["mode"] == "stream" else 0)
        if case["mode"] == "train":  # the backward reads the inputs and dy, and writes a gradient for each
            nbytes += e * (3 * s + 4 * sg) + 4 * bc * s + 2 * h0
        return {"bytes": float(nbytes), "flops": (19.0 if case["mode"] == "train" else 5.0) * e * n}
    train = case.get("mode", "train") == "train"
    flops, weights = _block_work(case)
    rows = case["batch"] * case["time"]
    if kind == "block":
        # the block's float32 input and output, and their gradients
        return {"bytes": (4.0 if train else 2.0) * 4 * rows * case["width"] + (2.0 if train else 1.0) * weights,
                "flops": (3.0 if train else 1.0) * flops}
    head = case["vocab"] * case["width"]
    return {"bytes": 2.0 * rows * case["vocab"] + 2.0 * (case["layers"] * weights + 4.0 * head),
            "flops": 3.0 * (case["layers"] * flops + 2.0 * rows * head)}


def tolerance(case):
    # a scan's outputs are rounded once to their type; float32 ones differ by the order of their sums
    if case["kind"] == "scan":
        return {"rel": {"f32": 2e-5, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]}
    if case["kind"] == "loss":
        return {"rel": 8e-3}
    # the block's 16-bit activations and gradients; in a model they pass through every layer
    return {"rel": 2e-2 if case["kind"] == "block" else 3e-2, "max": 0.8}


# ---- float64, plain torch ----------------------------------------------------------------------


def _affine64(f, w, x0):
    """x_t = f_t x_{t-1} + w_t for f [T, D, 1], w [T, D, N] from x0 [D, N]: chunks of L rows scanned from zero side by
    side, their carries in turn."""
    T, D, N = w.shape
    L = max(1, int(round(math.sqrt(T))))
    K = -(-T // L)
    x = torch.zeros(K * L, D, N, dtype=torch.float64, device=w.device)
    x[:T] = w
    p = torch.ones(K * L, D, 1, dtype=torch.float64, device=w.device)
    p[:T] = f
    x, p = x.view(K, L, D, N), p.view(K, L, D, 1)
    for t in range(1, L):
        x[:, t].addcmul_(p[:, t].expand(K, D, N), x[:, t - 1])
        p[:, t] *= p[:, t - 1]
    carry = x0
    for k in range(K):
        x[k].addcmul_(p[k].expand(L, D, N), carry.expand(L, D, N))
        carry = x[k, -1]
    return x.view(K * L, D, N)[:T]


def _scan64(u, fl, il, bm, cm, skip, h0):
    """One sequence ([T, D] streams, [T, N] B and C): y and the states."""
    f, i = torch.sigmoid(fl)[..., None], torch.sigmoid(il)
    x = _affine64(f, (i * u)[..., None] * bm[:, None, :], h0)
    return (x * cm[:, None, :]).sum(-1) + skip * u, x


def _scan64_grads(u, fl, il, bm, cm, skip, h0, dy):
    f, i = torch.sigmoid(fl), torch.sigmoid(il)
    _, x = _scan64(u, fl, il, bm, cm, skip, h0)
    dc = (x * dy[..., None]).sum(1)
    fr = torch.zeros_like(f)
    fr[1:] = f.flip(0)[:-1]
    g = _affine64(fr[..., None], (dy[..., None] * cm[:, None, :]).flip(0), torch.zeros_like(h0)).flip(0)
    prev = torch.cat([h0[None], x[:-1]])
    dfl = (g * prev).sum(-1) * f * (1 - f)
    dh0 = f[0][:, None] * g[0]
    dw = (g * bm[:, None, :]).sum(-1)
    db = (g * (i * u)[..., None]).sum(1)
    return i * dw + skip * dy, dfl, dw * u * i * (1 - i), db, dc, (dy * u).sum(0), dh0


class _Scan64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, u, fl, il, bm, cm):
        ctx.save_for_backward(u, fl, il, bm, cm)
        zero = torch.zeros(u.shape[-1], 1, dtype=u.dtype, device=u.device)
        return torch.stack([_scan64(u[k], fl[k], il[k], bm[k], cm[k], zero[:, 0], zero.expand(-1, bm.shape[-1]))[0]
                            for k in range(u.shape[0])])

    @staticmethod
    def backward(ctx, dy):
        u, fl, il, bm, cm = ctx.saved_tensors
        zero = torch.zeros(u.shape[-1], 1, dtype=u.dtype, device=u.device)
        got = [_scan64_grads(u[k], fl[k], il[k], bm[k], cm[k], zero[:, 0], zero.expand(-1, bm.shape[-1]), dy[k])[:5]
               for k in range(u.shape[0])]
        return tuple(torch.stack(v) for v in zip(*got))


def _norm64(x, w, eps=1e-5):
    return w * x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _conv64(x, w, b=None):
    k = w.shape[-1]
    xp = torch.nn.functional.pad(x, (0, 0, k - 1, 0))
    y = sum(xp[:, j:j + x.shape[1]] * w[:, 0, j] for j in range(k))
    return y if b is None else y + b


def _block64(x, p, at=""):
    w = {k[len(at):]: v for k, v in p.items() if k.startswith(at)}
    n = w["mixer.x_proj.weight"].shape[0] // 2
    xc, z = (_norm64(x, w["norm.weight"]) @ w["mixer.in_proj.weight"].t()).chunk(2, -1)
    h = torch.nn.functional.silu(_conv64(xc, w["mixer.conv1d.weight"], w["mixer.conv1d.bias"]))
    bm, cm = (h @ w["mixer.x_proj.weight"].t()).split(n, -1)
    fl, il = (h @ w[f"mixer.{s}_proj.weight"].t() + _conv64(h, w[f"mixer.{s}_conv.weight"]) + w[f"mixer.{s}_bias"]
              for s in "fi")
    cx = _Scan64.apply(h, fl, il, bm, cm)
    y = (cx / math.sqrt(n) + w["mixer.D"] * h) * torch.nn.functional.silu(z)
    return x + y @ w["mixer.out_proj.weight"].t()


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "scan":
        ins = [None if x is None else x.detach() for x in state["ins"]]
        train = case["mode"] == "train"
        skip, h0, dy = ins[5].double(), ins[6], state["dy"]
        ys, lasts, got = [], [], []
        for k in range(case["batch"]):
            one = [x[k].double() for x in ins[:5]]
            start = (torch.zeros(case["width"], case["state"], dtype=torch.float64, device="cuda") if h0 is None
                     else h0[k].double())
            y, x = _scan64(*one, skip, start)
            ys.append(y)
            lasts.append(x[-1].clone())
            del x
            if train:
                got.append(_scan64_grads(*one, skip, start, dy[k].double()))
        out = {"y": torch.stack(ys)}
        if case["mode"] == "stream":
            out["last"] = torch.stack(lasts)
        for j, name in enumerate(_SCAN_GRADS if train else ()):
            if j < 6 or h0 is not None:
                v = torch.stack([r[j] for r in got])
                out[name] = v.sum(0) if name == "dD_skip" else v
        return out
    if kind == "loss":
        logits, target = state["logits"].detach(), state["target"]
        rows, total, grad = case["rows"], 0.0, torch.empty_like(logits, dtype=torch.float64)
        for k in range(0, rows, 2048):
            x, y = logits[k:k + 2048].double(), target[k:k + 2048, None]
            lse = torch.logsumexp(x, 1, keepdim=True)
            total = total + (lse - x.gather(1, y)).sum()
            grad[k:k + 2048] = (torch.exp(x - lse)
                                - torch.zeros_like(x).scatter_(1, y, 1.0)) / rows
        return {"loss": total / rows, "dlogits": grad}
    train = case.get("mode", "train") == "train"
    p = {k: v.detach().double().requires_grad_(train) for k, v in state["model"].named_parameters()}
    if kind == "block":
        x = state["x"].detach().double().requires_grad_(train)
        y = _block64(x, p)
        if not train:
            return {"y": y}
        y.backward(state["dy"].double())
        return {"y": y.detach(), "dx": x.grad, **_take_grads(p.items())}
    x = torch.nn.functional.embedding(state["x"], p["embed.weight"])
    for j in range(case["layers"]):
        x = _block64(x, p, f"blocks.{j}.")
    logits = _norm64(x, p["norm.weight"]) @ p["embed.weight"].t()
    flat = logits.view(-1, case["vocab"])
    loss = (torch.logsumexp(flat, -1) - flat.gather(1, state["y"].view(-1, 1))[:, 0]).mean()
    loss.backward()
    return {"logits": logits.detach(), "loss": loss.detach(), **_take_grads(p.items())}
