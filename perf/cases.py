"""The workloads whose speed is tracked: what programs have this package do, through its public entry points.

A case names a path, a network and a batch:
  act     fc_forward: the logits of a batch (serving, rollouts, evaluation), float32 or bfloat16 states
  teach   fc_teach_step: forward, KL loss, backward and Adam, then the step's gradients fetched (fc_copy), as a learner
          that logs or exchanges them does
  play    NativeFlyActor without gradients, at any batch (a decision is a batch of 1)
  learn   NativeFlyActor with gradients, a loss in PyTorch, NativeAdam.step
  fly     FlyActor on the HopHip / FireHip kernels with PyTorch autograd (kernel "hip" or "cuda16")
  hop     HopHip alone: one hop's product and its backward
Networks: the synthetic 3-hop network of the benchmark (16,894 -> 46,393 -> 37,748 -> 1,332 rows, 2,992,734
connections) and its Erdos-Renyi control, whole (div 1) or with every count divided by div, as the tests use them; and
for the actors made from a graph file, a graph of the whole connectome's shape divided by div.
A network's connections depend on the case alone; weights, observations and teacher answers are drawn from the seed.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from flyguy_amd._lib import call, lib
from flyguy_amd.export import net_bytes, params_from_torch, structure
from flyguy_amd.fly import FlyActor
from flyguy_amd.fly_hip import HopHip
from flyguy_amd.fly_native import NativeFlyActor
from flyguy_amd.synth import WHOLE, scaled_3hop, whole_connectome

DEV = "cuda:0"
# the teaching trainer's default rates
LR, LR_NEURON, LR_PLUG, EMA = 3e-4, 1e-4, 3e-4, 0.999


def listed() -> list[dict]:
    return [
        # one decision of the full network through the C-ABI, padded to the library's tile: the latency of acting
        {"name": "act_32", "path": "act", "net": "lognormal", "div": 1, "batch": 32, "bf16": False},
        # a few hundred environments acting at once: an odd number of tiles
        {"name": "act_416", "path": "act", "net": "lognormal", "div": 1, "batch": 416, "bf16": False},
        # the benchmark's batch: evaluation and bulk inference
        {"name": "act_4096", "path": "act", "net": "lognormal", "div": 1, "batch": 4096, "bf16": False},
        # bulk inference with bfloat16 states
        {"name": "act_bf16_2048", "path": "act", "net": "lognormal", "div": 1, "batch": 2048, "bf16": True},
        # the teaching trainer's default batch
        {"name": "teach_512", "path": "teach", "net": "lognormal", "div": 1, "batch": 512, "bf16": False},
        # a ragged number of tiles on a graph of uniform in-degrees
        {"name": "teach_er_1056", "path": "teach", "net": "er", "div": 1, "batch": 1056, "bf16": False},
        # the benchmark's teaching step
        {"name": "teach_4096", "path": "teach", "net": "lognormal", "div": 1, "batch": 4096, "bf16": False},
        # the largest teaching step, bfloat16 states
        {"name": "teach_bf16_16384", "path": "teach", "net": "lognormal", "div": 1, "batch": 16384, "bf16": True},
        # one decision of an actor made from a graph file: the smallest call
        {"name": "play_1", "path": "play", "net": "connectome", "div": 8, "batch": 1},
        # a learner's minibatch of an odd size through PyTorch autograd and the library's Adam
        {"name": "learn_300", "path": "learn", "net": "connectome", "div": 8, "batch": 300},
        # FlyActor trained by PyTorch on the hop kernels: forward, KL, gradients of every parameter
        {"name": "fly_1024", "path": "fly", "net": "lognormal", "div": 1, "batch": 1024, "half": False},
        # one hop with binary16 states, forward and backward
        {"name": "hop_half_4096", "path": "hop", "net": "lognormal", "div": 1, "hop": 2, "batch": 4096, "half": True},
    ]


def draw(rng) -> dict:
    """A case of the same ranges, none of the listed ones."""
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    c = _draw(rng)
    while c in known:
        c = _draw(rng)
    return c


def _draw(rng) -> dict:
    def log_int(lo, hi):                        # (each whole number's share of the logarithm, the ends in full)
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))

    path = rng.choice(["act", "act", "teach", "teach", "play", "learn", "fly", "hop"])
    c = {"path": path}
    if path in ("play", "learn"):
        c.update(net="connectome", div=log_int(4, 32), batch=log_int(1, 2048))
        return c
    c.update(net=rng.choice(["lognormal", "er"]), div=log_int(1, 16))
    if path in ("act", "teach"):
        c["bf16"] = rng.random() < 0.35
        unit, most = (64, 16384) if c["bf16"] else (32, 4096)
        c["batch"] = unit * log_int(1, most // unit)
    else:
        c["half"] = rng.random() < 0.4
        c["batch"] = 32 * log_int(1, 64 if path == "fly" else 128)
        if path == "hop":
            c["hop"] = rng.randint(1, 3)
    return c


# ------------------------------------------------------------------------------------------------ networks
@functools.lru_cache(maxsize=4)
def _synthetic(kind: str, div: int) -> dict:
    return scaled_3hop(div, kind=kind)[0]


@functools.lru_cache(maxsize=2)
def _graph(div: int) -> dict:
    return whole_connectome(*(max(8, WHOLE[k] // div) for k in ("neurons", "connections", "sensory", "descending")))


def _params(s: dict, seed: int) -> list[np.ndarray]:
    """The seven weight arrays: strengths N(0, 1 / fan-in), gains and thresholds around their initial 1 and -4, the
    plug N(0, 1 / fan), the read-out N(0, 1 / descending rows)."""
    rng = np.random.default_rng([seed, 1])
    normal = lambda n: rng.standard_normal(n, dtype=np.float32)      # noqa: E731
    w = np.empty(s["n_w"], np.float32)
    for h in s["hop"]:
        fan_in = np.diff(h["crow"])
        w[h["widx"]] = normal(len(h["widx"])) / np.sqrt(np.repeat(fan_in, fan_in)).astype(np.float32)
    n = s["n_neurons"]
    return [w, 1 + 0.1 * normal(n), -4 + 0.2 * normal(n), normal(s["n_s"] * s["fan"]) / np.float32(math.sqrt(s["fan"])),
            0.1 * normal(s["n_s"]), normal(s["n_act"] * s["n_dn"]) / np.float32(math.sqrt(s["n_dn"])),
            0.1 * normal(s["n_act"])]


def _batch(s: dict, B: int, seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Observations and teacher logits on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    obs = torch.randn(B, s["obs_dim"], device=DEV, generator=g)
    return obs, 2 * torch.randn(B, s["n_act"], device=DEV, generator=g)


def _kl(logits: torch.Tensor, teacher: torch.Tensor) -> torch.Tensor:
    lt = torch.log_softmax(teacher, 1)
    return (lt.exp() * (lt - torch.log_softmax(logits, 1))).sum(1).mean()


def _actor(case: dict, seed: int) -> NativeFlyActor:
    """An actor as a program makes it from a graph file, then loaded with other weights (a checkpoint's)."""
    f = NativeFlyActor(_graph(case["div"]), 517, 90, hops=3, fan=16, max_batch=_tiles(case["batch"]))
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        f.w.mul_(8 * (0.5 + torch.rand(f.w.shape, generator=g)))
        f.gain.copy_(1 + 0.1 * torch.randn(f.gain.shape, generator=g))
        f.theta.copy_(-4 + 0.2 * torch.randn(f.theta.shape, generator=g))
        f.in_w.copy_(0.25 * torch.randn(f.in_w.shape, generator=g))
        f.in_b.copy_(0.1 * torch.randn(f.in_b.shape, generator=g))
        f.out.weight.copy_(torch.randn(f.out.weight.shape, generator=g) / math.sqrt(f.out.in_features))
        f.out.bias.copy_(0.1 * torch.randn(f.out.bias.shape, generator=g))
    return f


def _tiles(n: int) -> int:
    return -(-n // 32) * 32


# ------------------------------------------------------------------------------------------------ a state and a pass
class _Core:
    """A library handle with its weights set, freed with the state that holds it."""

    def __init__(self, s: dict, params: list[np.ndarray], batch: int, bf16: bool):
        raw = net_bytes(s)
        self.h = lib().fc_create_ex(raw, len(raw), batch, 1 if bf16 else 0)
        if not self.h:
            call("fc_create_ex")
        arrays = [torch.as_tensor(p).to(DEV) for p in params]
        for which in (0, 1):                    # the weights and their running average
            call("fc_copy", self.h, which, 1, self.pointers(arrays))

    @staticmethod
    def pointers(arrays):
        return (ctypes.c_void_p * 7)(*[a.data_ptr() for a in arrays])

    def __del__(self):
        if getattr(self, "h", None):
            lib().fc_free(self.h)


def prepare(case: dict, seed: int) -> dict:
    path, B = case["path"], case["batch"]
    st = {"path": path, "B": B}
    if path in ("act", "teach"):
        s = _synthetic(case["net"], case["div"])
        params = _params(s, seed)
        st["core"] = _Core(s, params, B, case["bf16"])
        st["obs"], st["teacher"] = _batch(s, B, seed)
        if path == "act":
            st["logits"] = torch.empty(B, s["n_act"], device=DEV)
        else:
            st["stats"] = torch.zeros(2, device=DEV)
            st["grads"] = [torch.empty(p.size, device=DEV) for p in params]
            st["grad_ptrs"] = _Core.pointers(st["grads"])
    elif path in ("play", "learn"):
        f = _actor(case, seed).to(DEV)
        st["actor"] = f
        st["obs"], st["teacher"] = _batch({"obs_dim": 517, "n_act": 90}, B, seed)
        if path == "learn":
            st["opt"] = f.native_adam(LR)
        else:
            with torch.no_grad():
                f(st["obs"][:1])                # (opens the library session, as a program's first decision does)
    elif path == "fly":
        s = _synthetic(case["net"], case["div"])
        f = FlyActor.from_structure(s, _params(s, seed)).to(DEV)
        f.kernel = "cuda16" if case["half"] else "hip"
        st["actor"] = f
        st["obs"], st["teacher"] = _batch(s, B, seed)
    else:
        s = _synthetic(case["net"], case["div"])
        h = s["hop"][case["hop"] - 1]
        put = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a, dtype=dt)).to(DEV)   # noqa: E731
        base = int(h["widx"].min())
        order = np.empty(len(h["widx"]), np.int64)
        order[h["widx"] - base] = np.arange(len(h["widx"]))
        st["index"] = (put(h["crow"], np.int64), put(h["col"], np.int32), put(h["tcrow"], np.int64),
                       put(h["tcol"], np.int32), put(order[h["twidx"] - base], np.int64))
        st["w"] = put(_params(s, seed)[0][h["widx"]], np.float32).requires_grad_()
        g = torch.Generator(device=DEV).manual_seed(seed)
        states = torch.relu(torch.randn(len(h["tcrow"]) - 1, B, device=DEV, generator=g))
        st["h"] = states.requires_grad_()
        gz = torch.randn(len(h["crow"]) - 1, B, device=DEV, generator=g) / B
        st["gz"] = gz * (torch.rand(gz.shape, device=DEV, generator=g) < 0.5)      # (half the neurons fired)
        st["half"] = case["half"]
    return st


def run(st: dict):
    path, B = st["path"], st["B"]
    if path == "act":
        call("fc_forward", st["core"].h, st["obs"].data_ptr(), B, st["logits"].data_ptr(), 0)
        return st["logits"]
    if path == "teach":
        h = st["core"].h
        call("fc_teach_step", h, st["obs"].data_ptr(), st["teacher"].data_ptr(), B, 1.0, LR, LR_NEURON, LR_PLUG, 0.0, EMA,
             st["stats"].data_ptr())
        call("fc_copy", h, 4, 0, st["grad_ptrs"])
        return {"stats": st["stats"], "grads": st["grads"]}
    f = st.get("actor")
    if path == "play":
        with torch.no_grad():
            return f(st["obs"])
    if path == "learn":
        st["opt"].zero_grad()
        logits = f(st["obs"])
        _kl(logits, st["teacher"]).backward()
        st["opt"].step()
        return {"logits": logits.detach(), "weights": [p.detach() for p in f.parameters()]}
    if path == "fly":
        logits = f(st["obs"])
        grads = torch.autograd.grad(_kl(logits, st["teacher"]), list(f.parameters()))
        return {"logits": logits.detach(), "grads": list(grads)}
    out = HopHip.apply(st["w"], st["h"], *st["index"], st["half"])
    gw, gh = torch.autograd.grad(out, (st["w"], st["h"]), st["gz"])
    return {"out": out.detach(), "gw": gw, "gh": gh}


# ------------------------------------------------------------------------------------------------ work
@functools.lru_cache(maxsize=16)
def _counts(net: str, div: int) -> tuple:
    """(rows per layer, connections per hop, re-drive rows per hop, strengths, neurons) of a case's network."""
    if net == "connectome":
        s = structure(NativeFlyActor(_graph(div), 517, 90, hops=3, fan=16, max_batch=32))
    else:
        s = _synthetic(net, div)
    return (list(s["sizes"]), [len(h["col"]) for h in s["hop"]], [int((h["drow"] >= 0).sum()) for h in s["hop"]],
            s["n_w"], s["n_neurons"])


def work(case: dict) -> dict:
    """A layer's states depend on all of the layer below, so each is written once and read once by every stage that needs
    it; connections (index and weight), observations, answers and parameters count once."""
    N, E, D, n_w, n_neurons = _counts(case["net"], case["div"])
    B = case["batch"]
    sz = 2 if case.get("bf16") or case.get("half") else 4
    if case["path"] == "hop":
        k = case["hop"]
        rows, src, e = N[k], N[k - 1], E[k - 1]
        # forward: h in, out written; backward: gz and h in, gh written; weights and indices per direction, gw written
        return {"bytes": 4 * B * (src + rows + rows + src + src) + 20 * e, "flops": 6 * e * B}
    fan, obs, act = 16, 517, 90
    params = n_w + 2 * n_neurons + (fan + 1) * N[0] + act * (N[-1] + 1)
    steps = sum(E) + fan * N[0] + act * N[-1]           # multiplications a sample
    states = sum(N) + sum(D)
    fwd = 4 * B * (obs + act) + 4 * params + 4 * (sum(E) + fan * N[0]) + 2 * sz * B * states
    if case["path"] in ("act", "play"):
        return {"bytes": fwd, "flops": 2 * steps * B}
    # backward: every layer's states once more, its gradient written and read, the gradients of the parameters
    bwd = sz * B * states + 2 * sz * B * states + 4 * params + 4 * B * obs + 4 * (sum(E) + fan * N[0])
    adam = 0 if case["path"] == "fly" else 36 * params
    return {"bytes": fwd + bwd + adam, "flops": 6 * steps * B}


# ------------------------------------------------------------------------------------------------ accuracy
def tolerance(case: dict) -> dict:
    if case["path"] in ("act", "play"):
        # float32 sums through four layers are 2e-7 off 64 bits; states rounded to bfloat16 at every layer 5e-3
        return {"rel": 2e-2 if case.get("bf16") else 1e-6}
    if case["path"] == "hop":
        return {"rel": 1.2e-3 if case["half"] else 1e-6}
    if case["path"] == "learn":
        # updated weights: where a gradient is near zero, Adam's first steps move by the whole rate either way
        return {"rel": 5e-6, "max": 2e-2}
    # gradients: a neuron within rounding of its threshold fires in one computation and not in another, and passes its
    # whole gradient or none
    return {"rel": 3e-2, "max": 0.99} if case.get("bf16") or case.get("half") else {"rel": 2e-3, "max": 0.99}


def _f64(a):
    return torch.as_tensor(np.asarray(a)).to(DEV, torch.float64)


def _long(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.int64)).to(DEV)


def _edge_dots(a: torch.Tensor, rows: torch.Tensor, b: torch.Tensor, cols: torch.Tensor) -> torch.Tensor:
    """sum over the batch of a[rows[e]] b[cols[e]] for every connection e, in pieces that fit the memory."""
    step = max(1, (1 << 28) // max(1, a.shape[1]))
    return torch.cat([(a[rows[i:i + step]] * b[cols[i:i + step]]).sum(1) for i in range(0, len(rows), step)])


class _Exact:
    """The network in float64 on plain PyTorch: forward of a piece of a batch and the gradients it adds."""

    def __init__(self, s: dict, params):
        self.s = s
        self.P = [_f64(p).reshape(-1) for p in params]
        W, self.gain, self.theta, in_w, self.in_b, out_w, self.out_b = self.P
        self.thr = torch.nn.functional.softplus(self.theta)
        self.out_w = out_w.view(s["n_act"], s["n_dn"])
        self.plug = (self.csr(s["in_crow"], s["in_col"], in_w, s["obs_dim"]), self.rows(s["in_crow"]), _long(s["in_col"]))
        self.hops = []
        for k, h in enumerate(s["hop"]):
            src, rows = s["sizes"][k], s["sizes"][k + 1]
            widx, twidx = _long(h["widx"]), _long(h["twidx"])
            drow = _long(h["drow"])
            at = torch.nonzero(drow >= 0).flatten()
            self.hops.append({"a": self.csr(h["crow"], h["col"], W[widx], src), "t": self.csr(h["tcrow"], h["tcol"], W[twidx], rows),
                              "row": self.rows(h["crow"]), "col": _long(h["col"]), "widx": widx, "nid": _long(h["nid"]),
                              "at": at, "drow": drow[at]})
        self.n0, self.dn = _long(s["n0"]), _long(s["dn_rows"])
        self.G = [torch.zeros_like(p) for p in self.P]

    @staticmethod
    def csr(crow, col, val, n):
        return torch.sparse_csr_tensor(_long(crow), _long(col), val, size=(len(crow) - 1, n))

    @staticmethod
    def rows(crow):
        return torch.repeat_interleave(torch.arange(len(crow) - 1, device=DEV), _long(np.diff(crow)))

    def forward(self, obs: torch.Tensor) -> torch.Tensor:
        self.x = obs.double().t().contiguous()
        fire = lambda z, nid: torch.relu(self.gain[nid, None] * z - self.thr[nid, None])      # noqa: E731
        drive = torch.sparse.mm(self.plug[0], self.x) + self.in_b[:, None]
        self.z, self.h = [drive], [fire(drive, self.n0)]
        for p in self.hops:
            z = torch.sparse.mm(p["a"], self.h[-1])
            z[p["at"]] += drive[p["drow"]]
            self.z.append(z)
            self.h.append(fire(z, p["nid"]))
        return (self.out_w @ self.h[-1][self.dn]).t() + self.out_b

    def backward(self, dl: torch.Tensor) -> None:
        gW, ggain, gtheta, gin_w, gin_b, gout_w, gout_b = self.G
        gout_w += (dl.t() @ self.h[-1][self.dn].t()).reshape(-1)
        gout_b += dl.sum(0)
        gh = torch.zeros_like(self.h[-1])
        gh[self.dn] = self.out_w.t() @ dl.t()
        gdrive = torch.zeros_like(self.z[0])

        def neurons(layer, nid):
            g = torch.where(self.h[layer] > 0, gh, 0)
            ggain[nid] += (g * self.z[layer]).sum(1)
            gtheta[nid] -= torch.sigmoid(self.theta[nid]) * g.sum(1)
            return g * self.gain[nid, None]

        for k in range(len(self.hops), 0, -1):
            p = self.hops[k - 1]
            gz = neurons(k, p["nid"])
            gdrive[p["drow"]] += gz[p["at"]]
            gW[p["widx"]] += _edge_dots(gz, p["row"], self.h[k - 1], p["col"])
            gh = torch.sparse.mm(p["t"], gz)
        gdrive += neurons(0, self.n0)
        gin_b += gdrive.sum(1)
        gin_w += _edge_dots(gdrive, self.plug[1], self.x, self.plug[2])

    def teach(self, obs, teacher) -> tuple[torch.Tensor, list[float]]:
        """Logits and loss sums of a batch; its gradients in self.G."""
        out, kl, agree, B = [], 0.0, 0, obs.shape[0]
        for i in range(0, B, 1024):
            lg, t = self.forward(obs[i:i + 1024]), teacher[i:i + 1024].double()
            ls, lt = torch.log_softmax(lg, 1), torch.log_softmax(t, 1)
            self.backward((ls.exp() - lt.exp()) / B)
            out.append(lg)
            kl += float((lt.exp() * (lt - ls)).sum())
            agree += int((lg.argmax(1) == t.argmax(1)).sum())
        return torch.cat(out), [kl, float(agree)]


def exact(case: dict, seed: int):
    path, B = case["path"], case["batch"]
    if path == "hop":
        st = prepare(case, seed)
        crow, col, tcrow, tcol, tperm = (a.long() for a in st["index"])
        w, h, gz = (st[k].detach().double() for k in ("w", "h", "gz"))
        row = torch.repeat_interleave(torch.arange(len(crow) - 1, device=DEV), crow.diff())
        a = torch.sparse_csr_tensor(crow, col, w, size=(len(crow) - 1, h.shape[0]))
        t = torch.sparse_csr_tensor(tcrow, tcol, w[tperm], size=(h.shape[0], len(crow) - 1))
        return {"out": torch.sparse.mm(a, h), "gw": _edge_dots(gz, row, h, col), "gh": torch.sparse.mm(t, gz)}
    if path in ("play", "learn"):
        f = _actor(case, seed)
        s = structure(f)
        e = _Exact(s, params_from_torch(f, s))
        obs, teacher = _batch(s, B, seed)
        if path == "play":
            return e.forward(obs)
        logits, _ = e.teach(obs, teacher)
        # the first Adam step: m / c1 = g, v / c2 = g^2
        lr = (LR, LR * f.lr_neuron, LR * f.lr_neuron) + (LR * f.lr_plug,) * 4
        new = [p - r * g / (g.abs() + 1e-8) for p, g, r in zip(e.P, e.G, lr)]
        w = _f64(f.w.detach())
        w[_long(s["wmap"])] = new[0]
        shapes = [p.shape for p in f.parameters()]
        return {"logits": logits, "weights": [v.reshape(n) for v, n in zip([w] + new[1:], shapes)]}
    s = _synthetic(case["net"], case["div"])
    e = _Exact(s, _params(s, seed))
    obs, teacher = _batch(s, B, seed)
    if path == "act":
        return torch.cat([e.forward(obs[i:i + 1024]) for i in range(0, B, 1024)])
    logits, stats = e.teach(obs, teacher)
    if path == "teach":
        return {"stats": torch.tensor(stats, dtype=torch.float64), "grads": e.G}
    shapes = [p.shape for p in FlyActor.from_structure(s).parameters()]
    return {"logits": logits, "grads": [g.reshape(n) for g, n in zip(e.G, shapes)]}
