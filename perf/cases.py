"""Timed cases of the framework: single layers, the row chain and whole training runs, through its public entry points.

A case is a dict of plain values with a "kind":
  linear   one Linear + ReLU layer: forward (act(x W^T + b)) or backward (dX under the previous layer's ReLU mask,
           the bias gradient, and the SGD update of W), f16 or f32, through Device.gemm and the reduce template
  softmax  softmax cross-entropy forward and backward over B rows of C logits, Device.softmax_ce
  chain    the permute / pad / shrink, softmax, RMS-normalise chain with its backward, Device.chain_step_noalloc
  convnet  a training run of the two-layer conv net (Trainer, replayed steps), then its loss and parameters are read
  mlp_ce   the same for the softmax-CE MLP, f32
  mlp3     the same for the three-layer MSE MLP in f16; the last step's gradients are read
  plan     one training step of the softmax-CE MLP as an item list replayed by a Plan: host arrays in, host arrays out

Sizes are the five training configurations of the benchmark and generic ones around them. Inputs are drawn on the GPU
from the seed. Device memory handed to Device.* calls is torch's; the library's own stream runs the work.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from anneal_amd import _lib as L
from anneal_amd import items as I
from anneal_amd.backend import Device, Trainer
from anneal_amd.executor import Plan

_STEPS = 100     # steps of one training run: a captured step is replayed 100 times between reads of the parameters
_LR = 1e-3
_DEVICE = None


def _dev() -> Device:
    """One device handle for the process, as a program holds it."""
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = Device(0)
    return _DEVICE


def listed():
    return [
        # the first layer of the f16 MLP at its training batch (4096 x 1024 -> 4096)
        {"name": "linear_f16_fwd_b4096", "kind": "linear", "dtype": "f16", "dir": "fwd", "M": 4096, "N": 4096, "K": 1024},
        # a wide f16 layer at a small batch: evaluation, and training with few samples per device
        {"name": "linear_f16_fwd_b32", "kind": "linear", "dtype": "f16", "dir": "fwd", "M": 32, "N": 4096, "K": 4096},
        # sizes that are no multiple of a tile: a last partial batch, 1000 classes, a width that is 8 past a multiple of 64
        {"name": "linear_f16_fwd_ragged", "kind": "linear", "dtype": "f16", "dir": "fwd", "M": 999, "N": 1000, "K": 2056},
        # backward of the f16 MLP's output layer (4096 x 4096 -> 1024): dX, the bias gradient and the weight update
        {"name": "linear_f16_bwd_b4096", "kind": "linear", "dtype": "f16", "dir": "bwd", "M": 4096, "N": 1024, "K": 4096},
        # backward of the dynamic-batch MLP's output layer (2048 -> 512) at batch 256, f32
        {"name": "linear_f32_bwd_b256", "kind": "linear", "dtype": "f32", "dir": "bwd", "M": 256, "N": 512, "K": 2048},
        # the loss of the dynamic-batch MLP at its largest batch
        {"name": "softmax_4096x512", "kind": "softmax", "B": 4096, "C": 512},
        # the reduce / movement chain at its benchmark size
        {"name": "chain_8192x4096", "kind": "chain", "R": 8192, "Cc": 4096},
        # the chain at a size that is no multiple of a tile
        {"name": "chain_3001x2052", "kind": "chain", "R": 3001, "Cc": 2052},
        # the small conv net's training run: 32 images of 28 x 28
        {"name": "convnet_b32", "kind": "convnet", "N": 32, "H": 28, "C1": 8, "C2": 16, "NC": 10},
        # the dynamic-batch MLP's training run at batch 256
        {"name": "mlp_ce_b256", "kind": "mlp_ce", "B": 256, "D": 512, "H": 2048, "C": 512},
        # the large f16 MLP's training run
        {"name": "mlp3_b4096", "kind": "mlp3", "B": 4096, "D0": 1024, "D1": 4096, "D2": 4096, "D3": 1024},
        # the small MLP's step as a captured item list fed from the host, the way a JIT replays it
        {"name": "plan_mlp_b64", "kind": "plan", "B": 64, "D": 784, "H": 128, "C": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 64 or 8, now and then any number."""
    w, pick = _log(rng, lo, hi), rng.random()
    step = 64 if pick < 0.5 else 8 if pick < 0.875 else 1
    return max(lo, w // step * step)


def draw(rng):
    pick = rng.random()
    if pick < 0.45:
        f16, fwd = rng.random() < 0.6, rng.random() < 0.5
        top = 8192 if f16 else 4096
        while True:
            m, n, k = _log(rng, 1, top), _width(rng, 64 if f16 else 10, top), _width(rng, 64 if f16 else 10, top)
            if m * n * k <= (4096 ** 3 if f16 else 4096 * 2048 * 1024):
                break
        return {"kind": "linear", "dtype": "f16" if f16 else "f32", "dir": "fwd" if fwd else "bwd", "M": m, "N": n, "K": k}
    if pick < 0.55:
        while True:
            b, c = _log(rng, 1, 16384), _log(rng, 2, 8192)
            if b * c <= 1 << 24:
                return {"kind": "softmax", "B": b, "C": c}
    if pick < 0.70:
        while True:
            r, c = _log(rng, 64, 16384), _log(rng, 64, 8192) // 4 * 4
            if r * c <= 1 << 25:
                return {"kind": "chain", "R": r, "Cc": c}
    if pick < 0.79:
        return {"kind": "convnet", "N": _log(rng, 1, 256), "H": 4 * rng.randint(3, 12), "C1": rng.randint(2, 16),
                "C2": rng.randint(4, 32), "NC": _log(rng, 2, 100)}
    if pick < 0.87:
        # Batches: up to 8, or up to 64 with a small model, any number; above, one whose last 32 rows close a 128-row
        # tile (the runs keep the hidden bias gradient as one partial row per 32 samples, laid out for those)
        b, d, h, c = _log(rng, 1, 2048), 8 * _log(rng, 4, 128), 8 * _log(rng, 4, 256), _log(rng, 2, 1024)
        if b <= 8:
            c = min(c, 512)
        elif not (b <= 64 and d <= 896 and h <= 128 and c <= 16):
            b = (b + 127) // 128 * 128 - rng.randint(0, 31)
        return {"kind": "mlp_ce", "B": b, "D": d, "H": h, "C": c}
    if pick < 0.93:
        # batch and output width in whole 256-wide tiles, for the same reason (the loss partials are per 32 x 32 block)
        w = lambda hi: 64 * (_log(rng, 256, hi) // 64)   # noqa: E731
        return {"kind": "mlp3", "B": 256 * rng.choice((1, 2, 3, 4, 5, 7, 8, 10, 12, 16)), "D0": w(1024), "D1": w(4096), "D2": w(4096),
                "D3": 256 * rng.randint(1, 4)}
    return {"kind": "plan", "B": _log(rng, 1, 256), "D": _width(rng, 32, 1024), "H": _width(rng, 32, 1024), "C": _log(rng, 2, 100)}


# ── inputs ─────────────────────────────────────────────────────────────────────

class _Buf:
    """Device memory as Device.* calls take it."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * std

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=self.g) * (hi - lo) + lo

    def labels(self, n, classes):
        return torch.randint(0, classes, (n,), device="cuda", generator=self.g, dtype=torch.int32)

    def kaiming(self, rows, cols, *rest):
        fan = cols * int(np.prod(rest)) if rest else cols
        b = math.sqrt(6.0 / fan)
        return self.uniform(rows, cols, *rest, lo=-b, hi=b)


def _inputs(case, seed):
    """The case's inputs as f32 (labels int32) tensors on the GPU; f16 values where the case is f16."""
    r, kind = _Rng(seed), case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        act = r.normal(M, K)
        if case["dir"] == "bwd":   # the previous layer's ReLU outputs; -0.0 marks a dead unit
            act = torch.where(act < 0, torch.full_like(act, -0.0), act)
        p = {"x": act, "W": r.normal(N, K, std=K ** -0.5), "b": r.normal(N, std=0.1)}
        if case["dir"] == "bwd":
            p["dy"] = r.normal(M, N)
        if case["dtype"] == "f16":
            p["W32"] = p["W"]
            p = {k: v if k == "W32" else v.half().float() for k, v in p.items()}
        return p
    if kind == "softmax":
        return {"z": r.normal(case["B"], case["C"], std=2.0), "labels": r.labels(case["B"], case["C"])}
    if kind == "chain":
        return {"X": r.normal(case["R"], case["Cc"]), "g": 1.0 + r.normal(case["Cc"], std=0.02)}
    if kind == "convnet":
        N, H, C1, C2, NC = (case[k] for k in ("N", "H", "C1", "C2", "NC"))
        return {"x": r.uniform(N, 1, H, H), "labels": r.labels(N, NC), "cw1": r.kaiming(C1, 1, 3, 3), "cb1": r.normal(C1, std=0.1),
                "cw2": r.kaiming(C2, C1, 3, 3), "cb2": r.normal(C2, std=0.1), "fw": r.kaiming(NC, C2 * (H // 4) ** 2), "fb": r.normal(NC, std=0.1)}
    if kind in ("mlp_ce", "plan"):
        B, D, H, K = (case[k] for k in ("B", "D", "H", "C"))
        return {"x": r.uniform(B, D, lo=-1.0), "labels": r.labels(B, K), "W1": r.kaiming(H, D), "b1": r.normal(H, std=0.01),
                "W2": r.kaiming(K, H), "b2": r.normal(K, std=0.01)}
    B, D0, D1, D2, D3 = (case[k] for k in ("B", "D0", "D1", "D2", "D3"))
    p = {"x": r.normal(B, D0).half().float(), "t": r.normal(B, D3).half().float()}
    for i, (a, b) in enumerate(((D0, D1), (D1, D2), (D2, D3)), 1):
        p["W%d" % i], p["b%d" % i] = r.normal(b, a, std=a ** -0.5), torch.zeros(b, device="cuda")
    return p


# ── the calls ──────────────────────────────────────────────────────────────────

class _Linear:
    def __init__(self, case, seed):
        self.c, p = case, _inputs(case, seed)
        f16 = case["dtype"] == "f16"
        self.dt, self.dev = (L.AH_F16 if f16 else L.AH_F32), _dev()
        cast = (lambda t: _Buf(t.half())) if f16 else (lambda t: _Buf(t.contiguous()))
        M, N, K = case["M"], case["N"], case["K"]
        new = lambda n, m, t=None: _Buf(torch.zeros(n, m, device="cuda", dtype=t or (torch.float16 if f16 else torch.float32)))   # noqa: E731
        self.x, self.W, self.b = cast(p["x"]), cast(p["W"]), cast(p["b"])
        if case["dir"] == "fwd":
            self.y = new(M, N)
            return
        self.dy, self.dx, self.db = cast(p["dy"]), new(M, K), _Buf(torch.zeros(N, device="cuda"))
        self.g = new(N, K, torch.float32)
        self.W32 = _Buf(p["W32"]) if f16 else self.W
        # the bias gradient's kernel, compiled or selected once
        self.k = C.c_void_p()
        key = "tmpl:reduce;dtype=%s;op=sum;axis=0;M=%d;N=%d;scale=%s" % (case["dtype"], M, N, I.f32_key(1.0 / M))
        L.check(self.dev.lib.ah_module_get(self.dev.h, key.encode(), b"kernel", C.byref(self.k)))
        self.ptrs = (C.c_void_p * 2)(self.db.ptr, self.dy.ptr)
        self.one = (C.c_uint32 * 3)(1, 1, 1)

    def run(self):
        d, M, N, K = self.dev, self.c["M"], self.c["N"], self.c["K"]
        if self.c["dir"] == "fwd":
            d.gemm(dtype=self.dt, epi=L.EPI_BIAS_RELU, ta=0, tb=0, M=M, N=N, K=K, A=self.x, B=self.W, lda=K, ldb=K,
                   C_out=self.y, ldc=N, bias=self.b)
            return self.y.t
        f16 = self.c["dtype"] == "f16"
        d.gemm(dtype=self.dt, epi=L.EPI_MASK, ta=0, tb=1, M=M, N=K, K=N, A=self.dy, B=self.W, lda=N, ldb=K, C_out=self.dx,
               ldc=K, aux=self.x, ldaux=K)
        L.check(d.lib.ah_launch(d.h, self.k, self.one, self.one, self.ptrs, 2, None, 0))
        d.gemm(dtype=self.dt, epi=L.EPI_SGD, ta=1, tb=1, M=N, N=K, K=M, A=self.dy, B=self.x, lda=N, ldb=K, ldc=K,
               scale=1.0 / M, W32=self.W32, W16=self.W if f16 else None, lr=1e-4, gout=self.g)
        out = {"dx": self.dx.t, "db": self.db.t, "dW": self.g.t, "W": self.W32.t}
        return dict(out, W16=self.W.t) if f16 else out


class _Softmax:
    def __init__(self, case, seed):
        p, self.c, self.dev = _inputs(case, seed), case, _dev()
        self.z, self.lab = _Buf(p["z"]), _Buf(p["labels"])
        self.dz, self.loss = _Buf(torch.zeros_like(p["z"])), _Buf(torch.zeros(1, device="cuda"))

    def run(self):
        self.dev.softmax_ce(self.z, self.lab, self.c["B"], self.c["C"], self.dz, self.loss)
        return {"dz": self.dz.t, "loss": self.loss.t}


class _Chain:
    def __init__(self, case, seed):
        p, self.c, self.dev = _inputs(case, seed), case, _dev()
        self.X, self.g, self.dX = _Buf(p["X"]), _Buf(p["g"]), _Buf(torch.zeros_like(p["X"]))
        self.dg, self.loss = _Buf(torch.zeros_like(p["g"])), _Buf(torch.zeros(1, device="cuda"))

    def run(self):
        self.dev.chain_step_noalloc(self.X, self.g, self.c["R"], self.c["Cc"], self.dX, self.dg, self.loss)
        return {"dX": self.dX.t, "dg": self.dg.t, "loss": self.loss.t}


class _Train:
    """A training run: _STEPS replayed steps, the last one keeping its gradients; then the parameters (f32) or the
    gradients (f16: the parameters move by less than their rounding in so few steps) are read with the loss."""

    KINDS = {"convnet": (L.TRAIN_CONVNET, ("N", "H", "C1", "C2", "NC"), "loss"),
             "mlp_ce": (L.TRAIN_MLP_CE, ("B", "D", "H", "C"), "loss"),
             "mlp3": (L.TRAIN_MLP3_F16, ("B", "D0", "D1", "D2", "D3"), "loss_sum")}

    def __init__(self, case, seed):
        kind, dims, self.loss = self.KINDS[case["kind"]]
        p, d = _inputs(case, seed), [case[k] for k in dims]
        self.t, self.B = Trainer(_dev(), kind, d, _LR), d[0]
        for k, v in p.items():
            self.t.set(k, v.cpu().numpy())
        self.sizes = {("d" if case["kind"] == "mlp3" else "") + k: v.numel() for k, v in p.items() if k not in ("x", "t", "labels")}

    def run(self):
        self.t.steps(self.B, _STEPS - 1, graph=True)
        self.t.step(self.B, store_grads=True)
        out = {k: self.t.get(k, n) for k, n in self.sizes.items()}
        out["loss"] = self.t.get(self.loss, 1)
        return out

    def __del__(self):
        if hasattr(self, "t"):
            self.t.close()


class _Plan:
    def __init__(self, case, seed):
        items, leaves, self.outs = I.mlp_ce(case["B"], case["D"], case["H"], case["C"])
        self.plan = Plan(_dev(), items, graph=True)
        self.ins = I.inputs(leaves, {k: v.cpu().numpy() for k, v in _inputs(case, seed).items()})

    def run(self):
        got = self.plan.run(self.ins)
        return {k: got[u] for k, u in self.outs.items()}

    def __del__(self):
        if hasattr(self, "plan"):
            self.plan.close()


_KINDS = {"linear": _Linear, "softmax": _Softmax, "chain": _Chain, "convnet": _Train, "mlp_ce": _Train, "mlp3": _Train, "plan": _Plan}


def prepare(case, seed):
    s = _KINDS[case["kind"]](case, seed)
    torch.cuda.synchronize()   # the inputs, made on torch's stream, are there before the library's stream reads them
    return s


def run(state):
    return state.run()


# ── work, tolerances, 64-bit values ────────────────────────────────────────────

def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        e = 2 if case["dtype"] == "f16" else 4
        if case["dir"] == "fwd":
            return {"bytes": e * (M * K + N * K + N + M * N), "flops": 2 * M * N * K}
        w = N * K * (2 + 4 + 4 + 4 + 2 if e == 2 else 4 + 4 + 4)   # W (f16 operand), master read and written, gradient, f16 copy
        return {"bytes": e * (M * N + 2 * M * K) + w + 4 * N, "flops": 4 * M * N * K}
    if kind == "softmax":
        return {"bytes": 8 * case["B"] * case["C"] + 4 * case["B"], "flops": 10 * case["B"] * case["C"]}
    if kind == "chain":
        return {"bytes": 8 * case["R"] * case["Cc"] + 8 * case["Cc"], "flops": 12 * case["R"] * case["Cc"]}
    if kind == "convnet":
        N, H, C1, C2, NC = (case[k] for k in ("N", "H", "C1", "C2", "NC"))
        F, H2 = C2 * (H // 4) ** 2, H // 2
        flops = N * (2 * 2 * 9 * C1 * H * H + 3 * 2 * 9 * C1 * C2 * H2 * H2 + 3 * 2 * F * NC)
        par = 10 * C1 + 9 * C1 * C2 + C2 + NC * F + NC
        return {"bytes": _STEPS * 4 * (N * H * H + N + 2 * par), "flops": _STEPS * flops}
    if kind in ("mlp_ce", "plan"):
        B, D, H, K = (case[k] for k in ("B", "D", "H", "C"))
        par, flops = H * D + H + K * H + K, 2 * B * (2 * D * H + 3 * H * K)
        n = _STEPS if kind == "mlp_ce" else 1
        return {"bytes": n * 4 * (B * D + B + 2 * par), "flops": n * flops}
    B, D0, D1, D2, D3 = (case[k] for k in ("B", "D0", "D1", "D2", "D3"))
    par, flops = D0 * D1 + D1 * D2 + D2 * D3, 2 * B * (2 * D0 * D1 + 3 * D1 * D2 + 3 * D2 * D3)
    return {"bytes": _STEPS * (2 * B * (D0 + D3) + 12 * par), "flops": _STEPS * flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # f16 results: a sum in another order moves single values by one or two f16 steps; f32: 32-bit sums
        return {"rel": 1e-3, "max": 8e-3} if case["dtype"] == "f16" else {"rel": 1e-5, "max": 1e-3}
    if kind == "softmax":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "chain":
        return {"rel": 2e-4, "max": 2e-2}   # dX of a column's maximum holds the rounding residue of the tie share
    if kind == "mlp3":
        return {"rel": 2e-2, "max": 0.99}   # f16 roundings and ReLU masks that flip travel through three layers
    if kind in ("convnet", "mlp_ce"):
        return {"rel": 2e-5, "max": 2e-3}   # 100 steps of f32 sums in another order
    return {"rel": 1e-5, "max": 1e-3}


def _ce(logits, labels):
    return torch.nn.functional.cross_entropy(logits, labels.long())


def _conv_net(p, x):
    def block(x, w, b):
        n, _, h, _ = x.shape
        z = torch.matmul(w.reshape(w.shape[0], -1), torch.nn.functional.unfold(x, 3, padding=1)) + b[:, None]
        return torch.relu(z).reshape(n, w.shape[0], h // 2, 2, h // 2, 2).amax((3, 5))
    h = block(block(x, p["cw1"], p["cb1"]), p["cw2"], p["cb2"])
    return h.reshape(x.shape[0], -1) @ p["fw"].T + p["fb"]


def _train64(case, p):
    """Gradient descent in 64 bits: what the run (or the plan's one step) reads at its end."""
    kind = case["kind"]
    names = [k for k in p if k not in ("x", "t", "labels")]
    x, w = p["x"].double(), {k: p[k].double() for k in names}
    for i in range(1 if kind == "plan" else _STEPS):
        w = {k: v.detach().requires_grad_() for k, v in w.items()}
        if kind == "convnet":
            loss = _ce(_conv_net(w, x), p["labels"])
        else:
            h = torch.relu(x @ w["W1"].T + w["b1"])
            h = h @ w["W2"].T + w["b2"]
            if kind == "mlp3":
                diff = torch.relu(h) @ w["W3"].T + w["b3"] - p["t"].double()
                loss = diff.square().mean()
            else:
                loss = _ce(h, p["labels"])
        g = torch.autograd.grad(loss, list(w.values()))
        w = {k: (v - _LR * d).detach() for (k, v), d in zip(w.items(), g)}
    out = {"d" + k: d for k, d in zip(names, g)} if kind in ("mlp3", "plan") else w
    out = {k: v.reshape(-1) for k, v in out.items()}
    out["loss"] = (diff.square().sum() if kind == "mlp3" else loss).detach().reshape(1)
    return out


def exact(case, seed):
    p, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        x, W, b = p["x"].double(), p["W"].double(), p["b"].double()
        if case["dir"] == "fwd":
            return torch.relu(x @ W.T + b)
        dy, M = p["dy"].double(), case["M"]
        g = dy.T @ x / M
        W2 = p["W32" if case["dtype"] == "f16" else "W"].double() - 1e-4 * g
        dead = torch.signbit(p["x"]) & (p["x"] == 0)
        out = {"dx": torch.where(dead, 0.0, dy @ W), "db": dy.sum(0) / M, "dW": g, "W": W2}
        return dict(out, W16=W2) if case["dtype"] == "f16" else out
    if kind == "softmax":
        z = p["z"].double().requires_grad_()
        loss = _ce(z, p["labels"])
        return {"dz": torch.autograd.grad(loss, z)[0], "loss": loss.detach().reshape(1)}
    if kind == "chain":
        X, g = p["X"].double().requires_grad_(), p["g"].double().requires_grad_()
        S = torch.softmax(X, 0)
        loss = (S * torch.rsqrt(S.square().mean(0) + 1e-6) * g).sum()
        dX, dg = torch.autograd.grad(loss, (X, g))
        return {"dX": dX, "dg": dg, "loss": loss.detach().reshape(1)}
    # A run with many ReLU units and pooling windows has some within a rounding of their threshold in every step; which
    # side they fall on moves the parameters by more than 32-bit sums do, so its parameters have no 64-bit value.
    if kind == "convnet" and case["N"] * case["H"] ** 2 * (case["C1"] + case["C2"] / 4) > 6e5:
        return None
    if kind == "mlp_ce" and case["B"] * case["H"] > 6e5:
        return None
    return _train64(case, p)
