"""The work a program has this package do, as measurable cases: windows of the recurrence (route,
forward sweep, backward with the carried state), a segment of carried windows, the fused cell
round, the state-gradient reverse sweep, the sparse round's operators and the trainer's passes. Each
case is a dict of sizes and options; :func:`prepare` makes what a program holds before the call,
:func:`run` is one pass through the public entry points, :func:`exact` the same pass in 64 bits by
plain torch.
"""

from __future__ import annotations

import torch

from hsn_amd import trainer, window
from hsn_amd.kernels import ops
from hsn_amd.kernels import window as window_kernels
from hsn_amd.state import CellGraphState
from hsn_amd.state_sweep import CellConstants, SweepRunner

F64 = torch.float64
IO = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _window(name, B, T, N, K, d, io="f32", **kw):
    case = dict(name=name, kind="window", B=B, T=T, N=N, M=1, K=K, d=d, io=io, norm=False,
                bias="none", cut=False, gate_mu=2.0, reset_p=1 / 256)
    case.update(kw)
    return case


def listed():
    return [
        # the smallest window a program runs (the gradient-check model): launches and host work
        _window("window_tiny", 2, 8, 16, 2, 16, reset_p=1 / 16),
        # the reference's own training recipe: few cells of eight units, the RMS candidate, unit
        # costs and a budget that cuts some positions' last slots
        _window("window_recipe", 32, 256, 32, 4, 64, M=8, norm=True, cut=True),
        # the headline training window
        _window("window_ref", 32, 256, 256, 8, 64),
        # the training window in bf16 storage with uneven cell popularity
        _window("window_bf16", 64, 512, 1024, 16, 64, "bf16", bias="normal", reset_p=1 / 128),
        # the largest window: many cells of heavily skewed popularity, bf16 storage
        _window("window_skewed", 256, 1024, 4096, 32, 64, "bf16", bias="zipf", reset_p=1 / 512),
        # two consecutive truncated-backprop windows, the state carried from the first into the
        # second and its gradient back into the first
        dict(_window("segment_tbptt", 128, 128, 512, 8, 128, gate_mu=3.0), kind="segment"),
        # the forward sweep without autograd: eight positions of the fused cell round, the state
        # carried from one to the next
        dict(name="round_model", kind="round", B=32, K=8, N=256, d=64, M=8, H=512, D=8, T=8),
        # one window of the state-gradient reverse sweep, bf16 products
        dict(name="sweep_model", kind="sweep", B=32, T=256, K=8, N=256, d=64, H=512, M=8, D=8,
             products="bf16"),
        # the unit bank on one position's pairs, forward and backward
        dict(name="mlp_position", kind="mlp", P=256, M=8, d=64, H=512, io="f32"),
        # the unit bank on a batch of positions' pairs in bf16
        dict(name="mlp_batch", kind="mlp", P=8192, M=8, d=64, H=512, io="bf16"),
        # one position's sparse round of a large batch as a training step: the four operators
        # forward, then their backwards
        dict(name="sparse_round", kind="sparse", B=256, K=16, N=1024, d=64, M=8, H=512, D=8),
        # the trainer's passes of one step over the model's 198 tensors: the gradients in, the
        # clip's scaling, AdamW and the weight average
        dict(name="trainer_model", kind="trainer", scale=1),
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["window"] * 6 + ["segment"] * 2 + ["round", "sweep", "mlp", "mlp", "sparse",
                                                          "trainer"])
    if kind in ("window", "segment"):
        while True:
            B, T, N = _log(rng, 1, 256), _log(rng, 8, 1024), _log(rng, 16, 4096)
            K = _log(rng, 1, min(32, N // 2))
            d = rng.choice([16, 24, 32, 40, 64, 64, 64, 96, 100, 128])
            M = rng.choice([1, 1, 1, 8])
            if B * T * K * d <= 2 ** 26 and B * T * N * M <= 2 ** 28 and B * N * d <= 2 ** 26:
                break
        case = _window("", B, T, N, K, d, rng.choice(["f32", "f32", "bf16"]), M=M,
                       norm=rng.random() < 0.3, bias=rng.choice(["none", "normal", "zipf"]),
                       cut=rng.random() < 0.2, gate_mu=rng.choice([2.0, 3.0]),
                       reset_p=rng.choice([0.0, 1 / 512, 1 / 128]))
        case["kind"] = kind
    elif kind in ("round", "sparse"):
        N = _log(rng, 16, 1024)
        case = dict(kind=kind, B=_log(rng, 1, 128 if kind == "round" else 256),
                    K=_log(rng, 1, min(16, N // 2)), N=N, d=rng.choice([16, 32, 64, 64, 128]), M=_log(rng, 1, 16),
                    H=rng.choice([64, 128, 256, 512]), D=_log(rng, 1, 12))
        if kind == "round":
            case["T"] = rng.randint(1, 8)
    elif kind == "sweep":
        N = _log(rng, 16, 512)
        case = dict(kind=kind, B=_log(rng, 1, 64), T=_log(rng, 8, 256),
                    K=_log(rng, 2, min(16, N // 2)), N=N, d=rng.choice([16, 32, 64, 64, 128]),
                    H=rng.choice([64, 128, 256, 512]), M=_log(rng, 1, 16), D=_log(rng, 1, 12),
                    products=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "mlp":
        case = dict(kind=kind, P=_log(rng, 1, 8192), M=_log(rng, 1, 16),
                    d=rng.choice([16, 32, 64, 64, 128]), H=rng.choice([64, 100, 256, 512]),
                    io=rng.choice(["f32", "f32", "bf16", "f16"]))
    else:
        case = dict(kind="trainer", scale=_log(rng, 1, 48))
    case.pop("name", None)
    return case


# --------------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, scale=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(scale).add_(mean)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _distinct_cells(g, *shape, N, K):
    return _rand(g, *shape, N).topk(K, dim=-1).indices


def _window_inputs(c, g):
    B, T, N, M, K, d, io = (c[k] for k in ("B", "T", "N", "M", "K", "d", "io"))
    dt = IO[io]
    bias = torch.zeros(N, device="cuda")
    if c["bias"] == "normal":
        bias = _randn(g, N, scale=0.5)
    elif c["bias"] == "zipf":
        bias = -1.1 * torch.log1p(torch.randperm(N, generator=g, device="cuda").float())
    logits = torch.empty(B, T, N, M, dtype=dt, device="cuda")
    for b in range(B):  # a row at a time: the fp32 draws of the largest window are 4 GB
        logits[b] = _randn(g, T, N, M) + bias[:, None]
    return {
        "logits": logits,
        "y": _randn(g, B, T, K, d).to(dt),
        "gate_pre": _randn(g, B, T, K, d, scale=0.5, mean=c["gate_mu"]).to(dt),
        "reset": _rand(g, B, T) < c["reset_p"],
        "d_q_pre": _randn(g, B, T, d).to(dt),
        "d_q_post": _randn(g, B, T, d).to(dt),
        "d_h_sel": _randn(g, B, T, K, d).to(dt),
    }


def _window_state(c, g):
    B, N, M, K, d = (c[k] for k in ("B", "N", "M", "K", "d"))
    h0 = _randn(g, B, N, d, scale=0.1)
    s = {"h0": h0, "q0": h0.mean(dim=1), "age0": torch.zeros(B, N, dtype=torch.int64, device="cuda"),
         "pos0": torch.zeros(B, dtype=torch.int64, device="cuda"),
         "d_h_T": _randn(g, B, N, d), "d_q_T": _randn(g, B, d),
         "cand_w": _randn(g, d, scale=0.1, mean=1.0)}
    if c["cut"]:  # unit costs about a K-th of the budget each
        s["cost"] = (0.85 / K) * (0.5 + _rand(g, M))
        s["cfg"] = window.RouteConfig(k=K, lambda_cost=0.05)
    else:
        s["cost"] = torch.full((M,), 1.0 / (N * M), device="cuda")
        s["cfg"] = window.RouteConfig(k=K)
    return s


def _graph(g, N, D):
    """A padded message graph: each cell's sources, about one in ten slots unused."""
    src = torch.randint(0, N, (N, D), generator=g, device="cuda")
    mask = _rand(g, N, D) < 0.9
    mask[:, 0] = True
    weights = torch.where(mask, torch.softmax(_randn(g, N, D), dim=1), torch.zeros((), device="cuda"))
    return torch.where(mask, src, torch.zeros_like(src)), mask, weights


class _Plain:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def _bank(g, M, d, H, dt=torch.float32):
    return {"W1": _randn(g, M, 4 * d, H, scale=(4 * d) ** -0.5).to(dt),
            "b1": _randn(g, M, H, scale=0.1).to(dt),
            "W2": _randn(g, M, H, d, scale=H ** -0.5).to(dt), "b2": _randn(g, M, d, scale=0.1).to(dt)}


def _round_inputs(c, g):
    B, K, N, d, M, H, D, T = (c[k] for k in ("B", "K", "N", "d", "M", "H", "D", "T"))
    src, _, edge_w = _graph(g, N, D)
    lin = {"V": _randn(g, d, d, scale=d ** -0.5), "gate_w": _randn(g, d, 4 * d, scale=(4 * d) ** -0.5),
           "gate_b": _randn(g, d, scale=0.2), "W_out": _randn(g, d, d, scale=d ** -0.5),
           "norm_w": _randn(g, 4 * d, scale=0.2, mean=1.0), "cand_w": _randn(g, d, scale=0.2, mean=1.0)}
    h = _rand(g, B, N, d) * 1.6 - 0.8
    valid = _rand(g, T, B, K) >= 1 / 16
    cells = torch.where(valid, _distinct_cells(g, T, B, N=N, K=K), torch.zeros((), dtype=torch.int64, device="cuda"))
    units = torch.where(valid, torch.randint(0, M, (T, B, K), generator=g, device="cuda"),
                        torch.zeros((), dtype=torch.int64, device="cuda"))
    return {"src": src, "edge_w": edge_w, "lin": lin, "bank": _bank(g, M, d, H), "h": h,
            "q": h.mean(dim=1), "age": torch.randint(0, 9, (B, N), generator=g, device="cuda"),
            "pos": torch.zeros(B, dtype=torch.int64, device="cuda"), "u": _randn(g, T, B, d),
            "eps": _randn(g, T, B, d), "cells": cells, "units": units, "valid": valid}


def _sweep_inputs(c, g):
    B, T, K, N, d, H, M, D = (c[k] for k in ("B", "T", "K", "N", "d", "H", "M", "D"))
    n = 4 * d
    src, mask, edge_w = _graph(g, N, D)
    consts = CellConstants(
        w_out=_randn(g, d, d, scale=d ** -0.5), cand_gain=_randn(g, d, scale=0.1, mean=1.0),
        cand_eps=1e-6, w2=_randn(g, M, H, d, scale=H ** -0.5),
        w1_state=_randn(g, M, 2 * d, H, scale=n ** -0.5), b1=_randn(g, M, H, scale=0.1),
        gate_state=_randn(g, d, 2 * d, scale=n ** -0.5), gate_bias=_randn(g, d, scale=0.1),
        norm_gain_state=_randn(g, 2 * d, scale=0.1, mean=1.0), in_dim=n,
        v=_randn(g, d, d, scale=d ** -0.5), edge_weights=edge_w, pad_src=src, activation="gelu",
        pad_mask=mask)
    hidden = _randn(g, B, T, K, H).to(IO[c["products"]])
    record = {"y": _randn(g, B, T, K, d), "alpha": torch.ones(B, T, K, device="cuda"), "hidden": hidden,
              "gate_pre": _randn(g, B, T, K, d), "m": _randn(g, B, T, K, d, scale=0.5),
              "rms": 0.5 + _rand(g, B, T, K)}
    args = (torch.tanh(_randn(g, B, T, K, d)), torch.sigmoid(_randn(g, B, T, K, d)),
            _randn(g, B, T, K, d, scale=0.5), _distinct_cells(g, B, T, N=N, K=K),
            torch.randint(0, M, (B, T, K), generator=g, device="cuda"), _rand(g, B, T, K) >= 1 / 16,
            _rand(g, B, T) < 1 / 64, N, _randn(g, B, T, d), _randn(g, B, T, d),
            _randn(g, B, T, K, d), None, record, consts)
    return args


def _sparse_inputs(c, g):
    B, K, N, d, M, H, D = (c[k] for k in ("B", "K", "N", "d", "M", "H", "D"))
    src, _, weights = _graph(g, N, D)
    h = _randn(g, B, N, d, scale=0.5)
    return {"indptr": torch.arange(N + 1, device="cuda") * D, "indices": src.reshape(-1),
            "a": weights.reshape(-1), "h": h, "q": h.mean(dim=1),
            "age": torch.randint(0, 9, (B, N), generator=g, device="cuda"), "u": _randn(g, B, d),
            "eps": _randn(g, B, d), "V": _randn(g, d, d, scale=d ** -0.5),
            "cells": _distinct_cells(g, B, N=N, K=K),
            "units": torch.randint(0, M, (B * K,), generator=g, device="cuda"),
            "valid": _rand(g, B, K) >= 1 / 16, "b": torch.sigmoid(_randn(g, B, K, d, mean=1.0)),
            "G": _randn(g, B, N, d), "gq": _randn(g, B, d), **_bank(g, M, d, H)}


#: The model's tensors: weights, biases and gains (198 of them, 1.97 M elements).
TRAINER_SIZES = [64 * 64] * 48 + [256 * 64] * 96 + [64] * 48 + [256 * 128] * 6
HYPER = dict(lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01, step=100)


def _mlp_inputs(c, g):
    P, M, d, H, dt = c["P"], c["M"], c["d"], c["H"], IO[c["io"]]
    return dict(_bank(g, M, d, H, dt), v=_randn(g, P, 4 * d).to(dt),
                unit=torch.randint(0, M, (P,), generator=g, device="cuda"),
                dout=_randn(g, P, d).to(dt))


def _trainer_inputs(c, g):
    total = sum(TRAINER_SIZES) * c["scale"]
    p = _randn(g, total, scale=0.05)
    return {"p": p, "raw": _randn(g, total, scale=1e-3), "m": _randn(g, total, scale=1e-3),
            "v": _randn(g, total, scale=1e-3).square_(), "ema": p + _randn(g, total, scale=1e-3),
            "clip": torch.rand(1, generator=g, device="cuda", dtype=F64) * 0.5 + 0.4}


def prepare(case, seed):
    c, g = case, _generator(seed)
    kind = c["kind"]
    if kind == "window":
        return {"case": c, **_window_inputs(c, g), **_window_state(c, g)}
    if kind == "segment":
        return {"case": c, "windows": [_window_inputs(c, g) for _ in range(2)],
                **_window_state(c, g)}
    if kind == "round":
        x = _round_inputs(c, g)
        lin, bank = x["lin"], x["bank"]
        weight = lambda w: _Plain(weight=torch.nn.Parameter(w))  # noqa: E731
        norm = lambda w: _Plain(weight=torch.nn.Parameter(w), eps=1e-6)  # noqa: E731
        x["cell"] = _Plain(
            d=c["d"], ablate_shared_u=False, cell_norm="rms", disabled_cells=(), cand_norm_kind="rms",
            V=weight(lin["V"]), norm=norm(lin["norm_w"]), W_out=weight(lin["W_out"]),
            gate=_Plain(weight=torch.nn.Parameter(lin["gate_w"]), bias=torch.nn.Parameter(lin["gate_b"])),
            cand_norm=norm(lin["cand_w"]), graph=_Plain(_pad_src=x["src"]),
            units=_Plain(activation_name="gelu", hidden=c["H"], **bank))
        x["state"] = CellGraphState.make(h=x["h"], q=x["q"], age=x["age"], pos=x["pos"])
        return {"case": c, **x}
    if kind == "sweep":
        args = _sweep_inputs(c, g)
        runner = SweepRunner()  # a training run keeps one; its first window captures the graph
        assert runner(*args, n_read=0) is not None
        return {"case": c, "args": args, "runner": runner}
    if kind == "mlp":
        return {"case": c, **_mlp_inputs(c, g)}
    if kind == "sparse":
        return {"case": c, **_sparse_inputs(c, g)}
    if kind == "trainer":
        x = _trainer_inputs(c, g)
        x["grad"] = torch.empty_like(x["raw"])
        sizes = [n * c["scale"] for n in TRAINER_SIZES]
        return {"case": c, **x, "lists": {k: list(torch.split(x[k], sizes))
                                         for k in ("p", "raw", "grad", "m", "v", "ema")}}
    raise ValueError(kind)


# --------------------------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------------------------

_SWEPT = ("slots", "theta", "q_pre", "q_post", "h_sel", "h_old", "h", "q", "h_max")


def _forward(c, s, w, h0, q0, age0, pos0, norm):
    return window.window_forward(w["logits"], w["y"], w["gate_pre"], w["reset"], h0, q0, age0, pos0,
                                 s["cost"], s["cfg"], **norm)


def _backward(c, w, out, d_h_T, d_q_T, norm):
    return window.backward(w["y"], w["gate_pre"], out["h_old"], out["slots"], w["reset"], c["N"],
                           w["d_q_pre"], w["d_q_post"], w["d_h_sel"], d_h_T, d_q_T, **norm)


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind in ("window", "segment"):
        norm = dict(cand_norm=True, cand_w=s["cand_w"]) if c["norm"] else {}
    if kind == "window":
        out = _forward(c, s, s, s["h0"], s["q0"], s["age0"], s["pos0"], norm)
        dy, dgate, d_h0, d_q0, d_w = _backward(c, s, out, s["d_h_T"], s["d_q_T"], norm)
        return dict(out, dy=dy, dgate=dgate, d_h0=d_h0, d_q0=d_q0, d_cand_w=d_w)
    if kind == "segment":
        at = [s[k] for k in ("h0", "q0", "age0", "pos0")]
        outs, grads, d_h, d_q = [], [], s["d_h_T"], s["d_q_T"]
        for w in s["windows"]:
            outs.append(_forward(c, s, w, *at, norm))
            at = [outs[-1][k] for k in ("h", "q", "age", "pos")]
        for w, out in zip(s["windows"][::-1], outs[::-1]):
            dy, dgate, d_h, d_q, d_w = _backward(c, w, out, d_h, d_q, norm)
            grads.append([dy, dgate, d_w])
        return {"outputs": [[o[k] for k in _SWEPT] for o in outs], "age": at[2], "pos": at[3],
                "grads": grads, "d_h0": d_h, "d_q0": d_q}
    if kind == "round":
        state = s["state"]
        sel = []
        for t in range(c["T"]):
            state, h_sel = window_kernels.cell_round(s["cell"], s["u"][t], s["eps"][t], state,
                                                     s["cells"][t], s["units"][t], s["valid"][t],
                                                     s["edge_w"])
            sel.append(h_sel)
        return {"h": state.h, "q": state.q, "age": state.age, "pos": state.pos, "h_sel": sel}
    if kind == "sweep":
        dc, db = s["runner"](*s["args"], n_read=0)
        return {"dc": dc, "db": db}
    if kind == "mlp":
        out, hidden = ops.mlp_op(s["v"], s["unit"], s["W1"], s["b1"], s["W2"], s["b2"])
        grads = ops.mlp_backward(s["v"], s["unit"], s["W1"], s["W2"], hidden, s["dout"])
        return {"out": out, "hidden": hidden, "grads": list(grads)}
    if kind == "sparse":
        B, K, N, d = c["B"], c["K"], c["N"], c["d"]
        with torch.no_grad():
            m = ops.messages_op(s["h"], s["indptr"], s["indices"], s["a"], s["V"], s["cells"])
            v = ops.gather_op(s["u"], s["eps"], s["h"], m, s["cells"]).view(B * K, 4 * d)
            f, hidden = ops.mlp_op(v, s["units"], s["W1"], s["b1"], s["W2"], s["b2"])
            cand = torch.tanh(f).view(B, K, d)
            h, q, age, old = ops.update_op(s["h"], s["q"], s["age"], s["cells"], s["valid"], cand, s["b"])
            dh, dq, dc, db = ops.update_backward(s["cells"], s["valid"], cand, s["b"], old, s["G"], s["gq"])
            df = (dc * (1 - cand * cand)).view(B * K, d)
            dv, dw1, db1, dw2, db2 = ops.mlp_backward(v, s["units"], s["W1"], s["W2"], hidden, df)
            du, de, dh_own, dm = ops.gather_backward(dv.view(B, K, 4 * d), s["cells"], N)
            dh_sources, da, dV = ops.messages_backward(s["h"], s["indptr"], s["indices"], s["a"], s["V"],
                                                       s["cells"], dm)
        return {"h": h, "q": q, "age": age, "old": old, "f": f,
                "grads": [dh, dh_own, dh_sources, dq, du, de, db, da, dV, dw1, db1, dw2, db2]}
    L = s["lists"]
    assert trainer.copy(L["grad"], L["raw"])  # the step's gradients, as the backward leaves them
    assert trainer.scale64(L["grad"], s["clip"])
    assert trainer.adamw(L["p"], L["grad"], L["m"], L["v"], **HYPER)
    assert trainer.lerp(L["ema"], L["p"], 0.01)
    return {"grad": s["grad"], "p": s["p"], "m": s["m"], "v": s["v"], "ema": s["ema"]}


# --------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct passes may be apart
# --------------------------------------------------------------------------------------------


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("window", "segment"):
        B, T, N, M, K, d = (c[k] for k in ("B", "T", "N", "M", "K", "d"))
        F = 4 if c["io"] == "f32" else 2
        route = N * M * F + 1 + 10 * K + 4
        fwd = 4 * K * d * F + 2 * d * F
        bwd = 6 * K * d * F + 2 * d * F
        state = B * (4 * N * d * 4 + 4 * d * 4 + 2 * N * 8)
        n = 2 if kind == "segment" else 1
        return {"bytes": n * (B * T * (route + fwd + bwd + 4) + state),
                "flops": n * B * T * (N * M + 40 * K * d)}
    if kind in ("round", "sparse"):
        B, K, N, d, M, H, D = (c[k] for k in ("B", "K", "N", "d", "M", "H", "D"))
        n = 4 * d
        units = min(M, B * K)
        weights = 4 * units * (n * H + H + H * d + d)
        state = 2 * B * (N * d * 4 + N * 8 + d * 4)
        slot = 2 * (n * H + H * d + d * d * (1 if kind == "sparse" else 2)
                    + (n * d if kind == "round" else 0) + D * d)
        if kind == "round":
            shared = 4 * (2 * d * d + n * d + n + 2 * d) + N * D * 12
            per = B * K * (21 + (D + 1) * d * 4 + d * 4) + 2 * B * d * 4
            return {"bytes": c["T"] * (state + weights + shared + per), "flops": c["T"] * B * K * slot}
        per = B * K * (17 + 2 * (D + 1) * d * 4 + 2 * n * 4 + 6 * d * 4) + 4 * B * d * 4
        return {"bytes": state + 2 * weights + 2 * B * N * d * 4 + per + N * D * 16,
                "flops": 3 * B * K * slot}
    if kind == "sweep":
        B, T, K, N, d, H, M, D = (c[k] for k in ("B", "T", "K", "N", "d", "H", "M", "D"))
        F = 2 if c["products"] == "bf16" else 4
        return {"bytes": B * T * (K * (9 * d * 4 + H * F + 29) + 2 * d * 4 + 1)
                + 4 * M * (3 * H * d + H) + N * D * 13,
                "flops": 2 * B * T * K * (d * H + (H + d) * 2 * d)}
    if kind == "mlp":
        P, M, d, H = c["P"], c["M"], c["d"], c["H"]
        F = 4 if c["io"] == "f32" else 2
        n, units = 4 * d, min(M, P)
        return {"bytes": F * (units * (2 * (n * H + H * d) + H + d) + M * (n * H + H * d + H + d)
                              + P * (3 * n + 2 * H + 2 * d)) + 16 * P,
                "flops": 6 * P * (n * H + H * d)}
    total = sum(TRAINER_SIZES) * c["scale"]
    return {"bytes": total * 4 * 10, "flops": total * 16}


def tolerance(case):
    c = case
    kind = c["kind"]
    if kind in ("window", "segment"):
        if c["io"] == "f32":
            return {"rel": 4e-6, "max": 4e-4, "differ": 0.0}
        return {"rel": 2e-3, "max": 3e-2, "differ": 0.0}  # a last bit of bf16 here and there
    if kind == "sweep":
        return {"rel": 3e-3 if c["products"] == "bf16" else 4e-6, "max": 0.1, "differ": 0.0}
    if kind == "mlp":
        return {"f32": {"rel": 2e-6, "max": 2e-4, "differ": 0.0},
                "f16": {"rel": 1e-3, "max": 2e-2, "differ": 0.0},
                "bf16": {"rel": 6e-3, "max": 1e-1, "differ": 0.0}}[c["io"]]
    if kind == "trainer":  # one correctly rounded operation after another
        return {"rel": 1e-7, "max": 1e-5, "differ": 0.0}
    return {"rel": 4e-6, "max": 4e-4, "differ": 0.0}


# --------------------------------------------------------------------------------------------
# the same passes in 64 bits
# --------------------------------------------------------------------------------------------


def _route_exact(c, logits, cost, cfg):
    """The decisions of every position: ``cells, units [B,T,K]``, ``valid`` and ``theta`` in 64
    bits. Scores are compared as the fp32 values they are."""
    B, T, N, M, K = (c[k] for k in ("B", "T", "N", "M", "K"))
    cells = torch.empty(B, T, K, dtype=torch.int64, device="cuda")
    units = torch.empty_like(cells)
    top = torch.empty(B, T, K + 1, device="cuda")
    index = N - 1 - torch.arange(N, device="cuda")
    rows = max(1, 2 ** 25 // (N * M * T))
    for b in range(0, B, rows):
        scores = logits[b:b + rows].float()
        if cfg.lambda_cost > 0:
            scores = scores - cfg.lambda_cost * cost
        score, unit = scores.max(dim=-1)  # ties: the first unit is checked below
        unit = (scores == score[..., None]).to(torch.int8).argmax(dim=-1) if M > 1 else unit
        bits = (score + 0.0).view(torch.int32)
        key = (bits ^ ((bits >> 31) & 0x7fffffff)).long() * 8192 + index
        best = key.topk(K + 1, dim=-1).indices
        cells[b:b + rows] = best[..., :K]
        units[b:b + rows] = unit.gather(-1, best[..., :K])
        top[b:b + rows] = score.gather(-1, best)
    spent = (cfg.shared_cost + (cfg.cell_overhead + cost[units]).double().cumsum(dim=-1)).float()
    valid = spent <= cfg.limit
    n = valid.sum(dim=-1, keepdim=True)
    lowest = top.gather(-1, (n - 1).clamp(min=0)).double().squeeze(-1)
    lowest = torch.where(n.squeeze(-1) > 0, lowest, torch.full_like(lowest, float("inf")))
    theta = 0.5 * (lowest + top.gather(-1, n).double().squeeze(-1))
    zero = torch.zeros_like(cells)
    return torch.where(valid, cells, zero), torch.where(valid, units, zero), valid, theta


def _candidate64(c, y, cand_w):
    y = y.to(F64)
    if not c["norm"]:
        return torch.tanh(y), None
    r = torch.rsqrt(y.square().mean(dim=-1, keepdim=True) + 1e-6)
    return torch.tanh(y * r * cand_w.to(F64)), r


def _forward64(c, w, cells, valid, h0, q0, cand_w):
    B, T, N, K, d = (c[k] for k in ("B", "T", "N", "K", "d"))
    cand, _ = _candidate64(c, w["y"], cand_w)
    gate = torch.sigmoid(w["gate_pre"].to(F64))
    h = torch.cat([h0, h0.new_zeros(B, 1, d)], dim=1)  # row N: the padded slots' own
    q = q0
    size = (B, T, K, d)
    h_sel, h_old = torch.empty(size, dtype=F64, device="cuda"), torch.empty(size, dtype=F64, device="cuda")
    q_pre, q_post = (torch.empty(B, T, d, dtype=F64, device="cuda") for _ in range(2))
    h_max = torch.empty(B, T, dtype=F64, device="cuda")
    resets = w["reset"].any(dim=0).tolist()
    for t in range(T):
        if resets[t]:
            h = h.masked_fill(w["reset"][:, t, None, None], 0)
            q = q.masked_fill(w["reset"][:, t, None], 0)
        q_pre[:, t] = q
        ok = valid[:, t, :, None]
        read = cells[:, t, :, None].expand(B, K, d)
        to = torch.where(ok, cells[:, t, :, None], N).expand(B, K, d)
        old = h.gather(1, read)
        new = torch.where(ok, (1 - gate[:, t]) * old + gate[:, t] * cand[:, t], 0)
        h = h.scatter(1, to, new)
        q = q + torch.where(ok, new - old, 0).sum(dim=1) / N
        h_old[:, t], h_sel[:, t], q_post[:, t] = old, h.gather(1, read), q
        h_max[:, t] = h[:, :N].abs().amax(dim=(1, 2))
    return dict(h_sel=h_sel, h_old=h_old, q_pre=q_pre, q_post=q_post, h=h[:, :N], q=q, h_max=h_max)


def _backward64(c, w, cells, valid, h_old, d_h_T, d_q_T, cand_w):
    B, T, N, K, d = (c[k] for k in ("B", "T", "N", "K", "d"))
    cand, r = _candidate64(c, w["y"], cand_w)
    gate = torch.sigmoid(w["gate_pre"].to(F64))
    A, R = torch.cat([d_h_T, d_h_T.new_zeros(B, 1, d)], dim=1), d_q_T
    dc, db = torch.empty_like(cand), torch.empty_like(cand)
    resets = w["reset"].any(dim=0).tolist()
    for t in reversed(range(T)):
        ok = valid[:, t, :, None]
        at = torch.where(ok, cells[:, t, :, None], N).expand(B, K, d)
        R = R + w["d_q_post"][:, t].to(F64)
        share = (R / N)[:, None, :]
        carried = A.gather(1, at) + w["d_h_sel"][:, t].to(F64)
        g = torch.where(ok, carried + share, 0)
        dc[:, t], db[:, t] = gate[:, t] * g, (cand[:, t] - h_old[:, t]) * g
        A = A.scatter(1, at, torch.where(ok, (1 - gate[:, t]) * carried - gate[:, t] * share, 0))
        R = R + w["d_q_pre"][:, t].to(F64)
        if resets[t]:
            A = A.masked_fill(w["reset"][:, t, None, None], 0)
            R = R.masked_fill(w["reset"][:, t, None], 0)
    dgate = db * gate * (1 - gate)
    dz = dc * (1 - cand * cand)
    d_w = None
    if c["norm"]:
        y = w["y"].to(F64)
        d_w = (dz * y * r).sum(dim=(0, 1, 2))
        dz = dz * cand_w.to(F64)
        dz = r * dz - r.pow(3) * y * (y * dz).mean(dim=-1, keepdim=True)
    return dz, dgate, A[:, :N], R, d_w


def _exact_window(c, g):
    w = _window_inputs(c, g)
    s = _window_state(c, g)
    cells, units, valid, theta = _route_exact(c, w.pop("logits"), s["cost"], s["cfg"])
    out = _forward64(c, w, cells, valid, s["h0"].to(F64), s["q0"].to(F64), s["cand_w"])
    dy, dgate, d_h0, d_q0, d_w = _backward64(c, w, cells, valid, out["h_old"], s["d_h_T"].to(F64),
                                             s["d_q_T"].to(F64), s["cand_w"])
    return dict(out, theta=theta, dy=dy, dgate=dgate, d_h0=d_h0, d_q0=d_q0, d_cand_w=d_w, cells=None,
                units=None, valid=None, refreshed=None, slots=None, age=None, pos=None)


def _exact_segment(c, g):
    ws = [_window_inputs(c, g) for _ in range(2)]
    s = _window_state(c, g)
    h, q = s["h0"].to(F64), s["q0"].to(F64)
    tapes, outs = [], []
    for w in ws:
        cells, _, valid, theta = _route_exact(c, w["logits"], s["cost"], s["cfg"])
        o = dict(_forward64(c, w, cells, valid, h, q, s["cand_w"]), theta=theta, slots=None)
        h, q = o["h"], o["q"]
        tapes.append((cells, valid, o["h_old"]))
        outs.append([o[k] for k in _SWEPT])
    A, R, grads = s["d_h_T"].to(F64), s["d_q_T"].to(F64), []
    for w, (cells, valid, h_old) in zip(ws[::-1], tapes[::-1]):
        dy, dgate, A, R, d_w = _backward64(c, w, cells, valid, h_old, A, R, s["cand_w"])
        grads.append([dy, dgate, d_w])
    return {"outputs": outs, "age": None, "pos": None, "grads": grads, "d_h0": A, "d_q0": R}


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x * 0.5 ** 0.5))


def _units64(x, unit, W):
    """``x[p] @ W[unit[p]]``."""
    out = x.new_empty(x.shape[0], W.shape[2])
    for j in range(W.shape[0]):
        at = (unit == j).nonzero().squeeze(1)
        out[at] = x[at] @ W[j].to(F64)
    return out


def _bank64(v, unit, bank):
    z = _units64(v, unit, bank["W1"]) + bank["b1"].to(F64)[unit]
    return _units64(_gelu64(z), unit, bank["W2"]) + bank["b2"].to(F64)[unit], z


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + 1e-6) * w


def _exact_round(c, g):
    x = _round_inputs(c, g)
    B, K, N, d, T = (c[k] for k in ("B", "K", "N", "d", "T"))
    lin = {k: w.to(F64) for k, w in x["lin"].items()}
    h, q = x["h"].to(F64), x["q"].to(F64)
    row = torch.arange(B, device="cuda")[:, None]
    sel = []
    for t in range(T):
        cells, valid = x["cells"][t], x["valid"][t]
        src = x["src"][cells]  # [B, K, D]
        m = (x["edge_w"].to(F64)[cells][..., None] * h[row[..., None], src]).sum(dim=2) @ lin["V"].T
        old = h[row, cells]
        wide = lambda a: a[t].to(F64)[:, None, :].expand(B, K, d)  # noqa: E731
        v = _rms64(torch.cat([wide(x["u"]), wide(x["eps"]), old, m], dim=-1), lin["norm_w"])
        b = torch.sigmoid(v @ lin["gate_w"].T + lin["gate_b"])
        f, _ = _bank64(v.reshape(B * K, 4 * d), x["units"][t].reshape(-1), x["bank"])
        y = _rms64(f.reshape(B, K, d) @ lin["W_out"].T, lin["cand_w"])
        new = (1 - b) * old + b * torch.tanh(torch.where(valid[..., None], y, 0))
        ok = valid[..., None]
        to = torch.where(ok, cells[..., None], N).expand(B, K, d)
        h = torch.cat([h, h.new_zeros(B, 1, d)], dim=1).scatter(1, to, torch.where(ok, new, 0))[:, :N]
        q = q + torch.where(ok, new - old, 0).sum(dim=1) / N
        sel.append(h[row, cells])
    return {"h": h, "q": q, "age": None, "pos": None, "h_sel": sel}


def _exact_sweep(c, g):
    (cand, gate, h_old, cells, units, valid, reset, N, d_q_pre, d_q_post, d_h_sel, _, rec,
     k) = _sweep_inputs(c, g)
    B, T, K, d, D = (c[k_] for k_ in ("B", "T", "K", "d", "D"))
    w = {f: getattr(k, f).to(F64) for f in ("w_out", "cand_gain", "w2", "w1_state", "b1", "gate_state",
                                            "gate_bias", "norm_gain_state", "v", "edge_weights")}
    P = B * K
    A = torch.zeros(B, N + 1, d, dtype=F64, device="cuda")
    R = torch.zeros(B, d, dtype=F64, device="cuda")
    dc, db = (torch.zeros(B, T, K, d, dtype=F64, device="cuda") for _ in range(2))
    M, H = c["M"], c["H"]
    w2_all = w["w2"].permute(2, 0, 1).reshape(d, M * H)  # [d, M H]: unit j's W2^T in its columns
    pick = torch.arange(P, device="cuda")
    one_of = torch.nn.functional.one_hot(units, M).to(F64)
    w1_all = w["w1_state"].permute(0, 2, 1).reshape(M * H, 2 * d)
    for t in reversed(range(T)):
        at64 = lambda a: a[:, t].to(F64)  # noqa: E731
        ok = valid[:, t, :, None]
        index = torch.where(ok, cells[:, t, :, None], N).expand(B, K, d)
        R = R + at64(d_q_post)
        A = A.scatter_add(1, index, torch.where(ok, at64(d_h_sel), 0))
        carried = A.gather(1, index)
        share = (R / N)[:, None, :]
        b, ct, ho = at64(gate), at64(cand), at64(h_old)
        total = torch.where(ok, carried + share, 0)
        dct, dbt = b * total, (ct - ho) * total
        dc[:, t], db[:, t] = dct, dbt
        y, hid = at64(rec["y"]), at64(rec["hidden"])
        dz = dct * (1 - ct * ct) * w["cand_gain"]
        rho = torch.rsqrt(y.square().mean(dim=-1, keepdim=True) + 1e-6)
        du = (rho * dz - rho.pow(3) * y * (y * dz).mean(dim=-1, keepdim=True)) @ w["w_out"]
        dg = dbt * b * (1 - b)
        act = (du.reshape(P, d) @ w2_all).view(P, M, H)[pick, units[:, t].reshape(-1)].view(B, K, H)
        slope = 0.5 * (1 + torch.erf(hid * 0.5 ** 0.5)) + hid * torch.exp(-0.5 * hid * hid) * 0.3989422804014327
        dh = act * slope
        dv = (one_of[:, t, :, :, None] * dh[:, :, None, :]).reshape(P, M * H) @ w1_all
        dv = dv.view(B, K, 2 * d) + dg @ w["gate_state"]
        sigma = (dh * (hid - w["b1"][units[:, t]])).sum(dim=-1)
        sigma = sigma + (dg * (at64(rec["gate_pre"]) - w["gate_bias"])).sum(dim=-1)
        r = at64(rec["rms"])[..., None]
        ds = r * (w["norm_gain_state"] * dv) - (r * r / k.in_dim) * torch.cat(
            [ho, at64(rec["m"])], dim=-1) * sigma[..., None]
        dvm = torch.where(ok, ds[..., d:] @ w["v"], 0)
        A = A.scatter(1, index, torch.where(ok, (1 - b) * carried - b * share + ds[..., :d], 0))
        safe = torch.where(valid[:, t], cells[:, t], torch.zeros_like(cells[:, t]))
        src = k.pad_src[safe].reshape(B, K * D, 1).expand(B, K * D, d)
        A = A.scatter_add(1, src, (w["edge_weights"][safe][..., None] * dvm[:, :, None, :])
                          .reshape(B, K * D, d))
        R = R + at64(d_q_pre)
        A = A.masked_fill(reset[:, t, None, None], 0)
        R = R.masked_fill(reset[:, t, None], 0)
    return {"dc": dc, "db": db}


def _exact_mlp(c, g):
    x = _mlp_inputs(c, g)
    v, unit, dout = x["v"].to(F64), x["unit"], x["dout"].to(F64)
    out, z = _bank64(v, unit, x)
    slope = 0.5 * (1 + torch.erf(z * 0.5 ** 0.5)) + z * torch.exp(-0.5 * z * z) * 0.3989422804014327
    dz = _units64(dout, unit, x["W2"].transpose(1, 2)) * slope
    dv = _units64(dz, unit, x["W1"].transpose(1, 2))
    act = _gelu64(z)
    grads = [[] for _ in range(4)]
    for j in range(c["M"]):
        at = (unit == j).nonzero().squeeze(1)
        for into, value in zip(grads, (v[at].T @ dz[at], dz[at].sum(0), act[at].T @ dout[at],
                                       dout[at].sum(0))):
            into.append(value)
    dw1, db1, dw2, db2 = (torch.stack(x_) for x_ in grads)
    return {"out": out, "hidden": z, "grads": [dv, dw1, db1, dw2, db2]}


def _exact_sparse(c, g):
    x = _sparse_inputs(c, g)
    B, K, N, d = (c[k] for k in ("B", "K", "N", "d"))
    leaf = lambda k: x[k].to(F64).requires_grad_(True)  # noqa: E731
    h_update, h_own, h_sources, q, u, eps, b, a, V, W1, b1, W2, b2 = (leaf(k) for k in (
        "h", "h", "h", "q", "u", "eps", "b", "a", "V", "W1", "b1", "W2", "b2"))
    row = torch.arange(B, device="cuda")[:, None]
    cells, valid = x["cells"], x["valid"][..., None]
    src = x["indices"].view(N, -1)[cells]  # [B, K, D]
    m = (a.view(N, -1)[cells][..., None] * h_sources[row[..., None], src]).sum(dim=2) @ V.T
    v = torch.cat([u[:, None].expand(B, K, d), eps[:, None].expand(B, K, d), h_own[row, cells], m], dim=-1)
    v = v.reshape(B * K, 4 * d)
    f = torch.zeros(B * K, d, dtype=F64, device="cuda")
    for j in range(c["M"]):
        at = (x["units"] == j).nonzero().squeeze(1)
        f = f.index_put((at,), _gelu64(v[at] @ W1[j] + b1[j]) @ W2[j] + b2[j])
    old = h_update[row, cells]
    change = torch.where(valid, b * (torch.tanh(f).view(B, K, d) - old), 0)
    h = h_update.scatter_add(1, cells[..., None].expand(B, K, d), change)
    new_q = q + change.sum(dim=1) / N
    grads = torch.autograd.grad([h, new_q], [h_update, h_own, h_sources, q, u, eps, b, a, V, W1, b1, W2, b2],
                                [x["G"].to(F64), x["gq"].to(F64)])
    return {"h": h.detach(), "q": new_q.detach(), "age": None,
            "old": torch.where(valid, old.detach(), 0), "f": f.detach(), "grads": list(grads)}


def _exact_trainer(c, g):
    x = {k: v.to(F64) for k, v in _trainer_inputs(c, g).items()}
    lr, b1, b2, step = (HYPER[k] for k in ("lr", "beta1", "beta2", "step"))
    grad = x["raw"] * x["clip"]
    m = x["m"] + (1 - b1) * (grad - x["m"])
    v = b2 * x["v"] + (1 - b2) * grad * grad
    p = x["p"] * (1 - lr * HYPER["weight_decay"])
    p = p - lr / (1 - b1 ** step) * m / ((v / (1 - b2 ** step)).sqrt() + HYPER["eps"])
    return {"grad": grad, "p": p, "m": m, "v": v, "ema": x["ema"] + 0.01 * (p - x["ema"])}


def exact(case, seed):
    with torch.enable_grad():
        return {"window": _exact_window, "segment": _exact_segment, "round": _exact_round,
                "sweep": _exact_sweep, "mlp": _exact_mlp, "sparse": _exact_sparse,
                "trainer": _exact_trainer}[case["kind"]](case, _generator(seed))
