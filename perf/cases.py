"""What a user of the evaluator has it do, as cases that can be timed and checked.

The network is the full-size one (166,700 neurons, about 10.5M synapses, 17,937 sensory and 2,333 output neurons) on
two wirings: "uniform", the package's synthetic graph, and "typed", whose in-degrees are heavy-tailed and alike among
neighbours, as in a connectome that numbers its neurons by cell type.  A program builds its network once and then
meets new boards, so the networks are made once per process; boards, drives, targets and snapshots are drawn from the
seed of each state.

Kinds of work ("what"):
* model      FlyChessNet.forward in evaluation: boards -> policy and WDL logits.
* io         ConnectomeRNN.forward_io: the recurrence alone, through the light cone.
* literal    ConnectomeRNN.forward: the recurrence over every neuron.
* evaluator  Evaluator(x, rows, cols): host boards in, host answers out (legal moves' logits, or the whole policy).
* train      FlyChessNet.forward under autograd, the training loss and its backward: logits and every gradient.
* refresh    load_weights of a new snapshot, then the first forward with it.
"""

from __future__ import annotations

import copy
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "alpha-fly_amd"))

from chessfly.encoding import N_BASE, N_FEATURES, N_MOVES, move_squares  # noqa: E402
from chessfly.model import Evaluator, FlyChessNet, ModelConfig, RunningNorm, load_weights  # noqa: E402
from chessfly.synthetic import FULL, synthetic_connectome  # noqa: E402

DEV = "cuda:0"
GAIN = 5.0                     # ModelConfig.input_gain
DTYPES = {"f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # one position at a time: a game against the engine, an analysis board
        {"name": "one position", "what": "model", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False,
         "batch": 1},
        # a search with a few games left, or a small match: the recurrence on an odd handful of positions
        {"name": "handful", "what": "io", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False, "batch": 21},
        # an arena's or a test suite's batch, with the default number of steps
        {"name": "arena", "what": "io", "graph": "uniform", "dtype": "f16", "steps": 4, "planes": False, "batch": 187},
        # self-play: one leaf of each of 1,120 games, the headline workload
        {"name": "self-play", "what": "model", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False,
         "batch": 1120},
        # the largest batch of the batch sweep
        {"name": "large batch", "what": "model", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False,
         "batch": 4096},
        # hub neurons and the attack-plane features, on an odd batch
        {"name": "hubs", "what": "model", "graph": "typed", "dtype": "f16", "steps": 6, "planes": True, "batch": 517},
        # the float32 light cone: evaluation where half precision is not wanted
        {"name": "float32 cone", "what": "io", "graph": "uniform", "dtype": "f32", "steps": 6, "planes": False,
         "batch": 256},
        # every neuron at every step in float32, 64 positions: probing the network's activity
        {"name": "literal", "what": "literal", "graph": "uniform", "dtype": "f32", "steps": 6, "planes": False,
         "batch": 64},
        # the search's own call: host boards up, the legal moves' logits and the values down
        {"name": "search call", "what": "evaluator", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False,
         "batch": 480, "lazy": False},
        # a training step at the trainer's batch
        {"name": "training", "what": "train", "graph": "uniform", "dtype": "f32", "steps": 6, "planes": False,
         "batch": 256},
        # the ragged last batch of a pass over the replay buffer
        {"name": "training, ragged", "what": "train", "graph": "uniform", "dtype": "f32", "steps": 6, "planes": False,
         "batch": 67},
        # a self-play worker taking the trainer's new snapshot
        {"name": "new snapshot", "what": "refresh", "graph": "uniform", "dtype": "f16", "steps": 6, "planes": False,
         "batch": 128},
    ]


def draw(rng):
    def size(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    what = rng.choice(["model", "model", "io", "io", "literal", "evaluator", "train", "refresh"])
    case = {"what": what, "graph": rng.choice(["uniform", "uniform", "typed"]), "dtype": "f16",
            "steps": rng.choice([4, 6, 6]), "planes": False}
    if what == "model":
        case["dtype"] = rng.choice(["f16", "f16", "f32"])
        case["planes"] = rng.random() < 0.25
        case["batch"] = size(1, 4096 if case["dtype"] == "f16" and case["graph"] == "uniform" else 1500)
    elif what == "io":
        case["dtype"] = rng.choice(["f16", "f32"])
        case["batch"] = size(1, 2048 if case["dtype"] == "f16" else 1024)
    elif what == "literal":
        case["dtype"] = "f32"
        case["batch"] = size(1, 256)
    elif what == "evaluator":
        case["lazy"] = rng.random() < 0.5
        case["batch"] = size(1, 2048)
    elif what == "train":
        case["dtype"] = "f32"
        case["batch"] = size(8, 256)
    else:
        case["batch"] = size(1, 512)
    return case


# ---- the networks ---------------------------------------------------------------------------------------------

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1_000_003 + salt) % (1 << 62))


@functools.lru_cache(maxsize=None)
def _graph(kind):
    """The Connectome, and the weight scale that gives the signed weight matrix a spectral radius of 0.9."""
    conn = synthetic_connectome()
    if kind == "typed":
        n = conn.n_neurons
        g = _gen(7, 1)
        types = torch.randn(n // 80 + 1, generator=g, device=DEV).repeat_interleave(80)[:n]     # runs of 80 neurons
        raw = torch.exp(types.double() + 0.5 * torch.randn(n, generator=g, device=DEV).double())
        deg = (raw * (FULL.edges / raw.sum())).round().long().clamp_max(9193)
        fame = torch.exp(torch.randn(n, generator=g, device=DEV).double()).cumsum(0)
        post = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
        pre = torch.searchsorted(fame / fame[-1], torch.rand(post.numel(), generator=g, device=DEV).double())
        pre = pre.clamp_max(n - 1)
        key = torch.unique((post * n + pre)[post != pre])                       # (post, pre) order, no repeats
        post, pre = key // n, key % n
        u = torch.rand(key.numel(), generator=g, device=DEV).double()
        syn = 1 + torch.floor(torch.log1p(-u) / math.log(0.75))                 # Geometric(1/4) on 1, 2, ...
        sign = torch.where(torch.rand(n, generator=g, device=DEV) < 0.6, 1.0, -1.0)
        conn = dataclasses.replace(conn, pre=pre.cpu(), post=post.cpu(), syn_count=syn.float().cpu(),
                                   sign=sign[pre].cpu())
    n = conn.n_neurons
    crow = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    crow[1:] = torch.bincount(conn.post.to(DEV), minlength=n).cumsum(0)
    mat = torch.sparse_csr_tensor(crow, conn.pre.to(DEV), (conn.sign * conn.weight).double().to(DEV), (n, n))
    v = torch.ones(n, 1, dtype=torch.float64, device=DEV)
    grown = 0.0
    for i in range(60):
        v = mat @ v
        norm = float(v.norm())
        grown += math.log(norm) if i >= 30 else 0.0
        v /= norm
    return conn, float(f"{0.9 / math.exp(grown / 30):.4g}")


def _draw_weights(net, seed):
    """A network's trainable state, drawn from the seed, as a state dict on the GPU."""
    g = _gen(seed, 2)
    state = {}
    for name, p in net.state_dict().items():
        r = torch.randn(p.shape, generator=g, device=DEV) if p.dtype == torch.float32 else None
        if name == "brain.log_gain":
            state[name] = 0.1 * r
        elif name == "brain.bias":
            state[name] = 0.1 + 0.05 * r
        elif name == "brain.alpha_logit":
            state[name] = r
        elif name.startswith("norm."):
            state[name] = p.clone()
        elif name == "encoder.weight":
            state[name] = r / math.sqrt(N_BASE)
        elif name == "encoder.bias":
            state[name] = r / math.sqrt(N_BASE)
        else:
            state[name] = r / math.sqrt(len(net.out_idx))
    return state


@functools.lru_cache(maxsize=None)
def _template(kind):
    conn, scale = _graph(kind)
    net = FlyChessNet(conn, ModelConfig(weight_scale=scale)).to(DEV)
    load_weights(net, _draw_weights(net, 0))
    return net.eval()


@functools.lru_cache(maxsize=None)
def _net(kind, steps, planes, dtype, role):
    """The network of a program that does `role` (one that trains or takes snapshots has its own)."""
    net = copy.deepcopy(_template(kind))
    net.cfg = dataclasses.replace(net.cfg, steps=steps, attack_planes=planes)
    net.infer_dtype = DTYPES[dtype]
    return net


@functools.lru_cache(maxsize=None)
def _evaluator(kind, steps, planes, dtype):
    return Evaluator(_net(kind, steps, planes, dtype, "play"), DEV)


# ---- inputs ----------------------------------------------------------------------------------------------------

def _boards(case, seed):
    """(batch, N_FEATURES) float32 boards: 20 to 40 of the base features set, and about a third of the attack planes
    where the network reads them."""
    g = _gen(seed, 3)
    b = case["batch"]
    count = torch.randint(20, 41, (b, 1), generator=g, device=DEV)
    rank = torch.rand(b, N_BASE, generator=g, device=DEV).argsort(1).argsort(1)
    x = torch.zeros(b, N_FEATURES, device=DEV)
    x[:, :N_BASE] = (rank < count).float()
    if case["planes"]:
        x[:, N_BASE:] = (torch.rand(b, N_FEATURES - N_BASE, generator=g, device=DEV) < 0.33).float()
    return x


def _drive(net, x, dtype):
    """The drive of the input neurons for boards x, (n_in, batch)."""
    k = N_FEATURES if net.cfg.attack_planes else N_BASE
    return (F.linear(x[:, :k], net.encoder.weight[:, :k], net.encoder.bias) * GAIN).to(dtype).T.contiguous()


def _legal(case, seed):
    """About 32 legal moves per board, as (rows, cols) index arrays; how many is the batch's, which ones the seed's."""
    per = np.random.default_rng(case["batch"]).integers(1, 64, case["batch"])
    rows = np.repeat(np.arange(case["batch"]), per)
    return rows, np.random.default_rng([int(seed) % (1 << 31), 11]).integers(0, N_MOVES, rows.size)


def _targets(case, seed):
    """A visit distribution over about 30 legal moves per position, and a result per position."""
    g = _gen(seed, 4)
    b = case["batch"]
    legal = torch.rand(b, N_MOVES, generator=g, device=DEV) < 30 / N_MOVES
    legal[:, 0] = True
    pi = torch.where(legal, torch.rand(b, N_MOVES, generator=g, device=DEV), 0.0)
    return pi / pi.sum(1, keepdim=True), legal, torch.randint(0, 3, (b,), generator=g, device=DEV)


def _loss(logits, wdl_logits, pi, legal, wdl):
    logp = logits.masked_fill(~legal, -1e9).log_softmax(-1)
    return -(pi * logp).sum(-1).mean() + F.cross_entropy(wdl_logits, wdl)


@torch.no_grad()
def prepare(case, seed):
    what = case["what"]
    key = (case["graph"], case["steps"], case["planes"], case["dtype"])
    x = _boards(case, seed)
    dtype = DTYPES[case["dtype"]]
    if what == "model":
        return {"what": what, "net": _net(*key, "play"), "x": x.to(dtype)}
    if what == "io":
        net = _net(*key, "play")
        return {"what": what, "net": net, "u": _drive(net, x, dtype)}
    if what == "literal":
        net = _net(*key, "play")
        u = torch.zeros(net.brain.n, case["batch"], device=DEV)
        u[net.in_idx] = _drive(net, x, torch.float32)
        return {"what": what, "net": net, "u": u, "steps": case["steps"]}
    if what == "evaluator":
        rows, cols = (None, None) if case["lazy"] else _legal(case, seed)
        return {"what": what, "evaluate": _evaluator(*key), "x": x.half().cpu().numpy(), "rows": rows, "cols": cols}
    if what == "train":
        shared = _net(*key, "train")
        net = copy.copy(shared)                         # the shared weights with running statistics of its own
        net._modules = dict(shared._modules)
        net.norm = RunningNorm(len(net.out_idx)).to(DEV)
        net.train()
        return {"what": what, "net": net, "x": x, "targets": _targets(case, seed)}
    net = _net(*key, "refresh")
    return {"what": what, "net": net, "snapshot": _draw_weights(net, seed), "x": x.to(dtype)}


def run(state):
    what = state["what"]
    if what == "train":
        net = state["net"]
        net.zero_grad(set_to_none=True)
        logits, wdl = net(state["x"])
        loss = _loss(logits, wdl, *state["targets"])
        loss.backward()
        return {"loss": loss.detach(), "logits": logits.detach(), "wdl": wdl.detach(),
                "grads": {k: p.grad for k, p in net.named_parameters()}}
    with torch.no_grad():
        if what == "evaluator":
            return state["evaluate"](state["x"], state["rows"], state["cols"])
        net = state["net"]
        if what == "literal":
            return net.brain(state["u"].clone(), state["steps"])        # the call adds the bias to its argument
        if what == "io":
            return net.brain.forward_io(state["u"], net.in_idx, net.out_idx, net.cfg.steps)
        if what == "refresh":
            load_weights(net, state["snapshot"])
        return net(state["x"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

# Synapses that some output's light cone visits, summed over the steps (LightCone.edge_visits of the two graphs), and
# the synapses of each graph.
VISITS = {("uniform", 6): 27_085_788, ("uniform", 4): 6_134_787, ("typed", 6): 25_839_442, ("typed", 4): 5_566_129}
SYNAPSES = {"uniform": 10_494_794, "typed": 10_481_388}


def work(case):
    """Bytes: the synapses (index and weight) and the dense maps' weights read once, inputs read and outputs written
    once.  Operations: two for each visited synapse and position, and the dense maps' products; a training step has
    three products where an evaluation has one, and writes a gradient for each weight."""
    n, n_in, n_out, b, what = FULL.n, FULL.n_sensory, FULL.n_output, case["batch"], case["what"]
    visits, synapses = VISITS[case["graph"], case["steps"]], SYNAPSES[case["graph"]]
    size = 2 if case["dtype"] == "f16" else 4
    k = N_FEATURES if case["planes"] else N_BASE
    dense = n_in * k + n_out * (N_MOVES + 128 + 3)
    brain = 8 * synapses + 8 * n
    if what == "io":
        return {"bytes": brain + b * (n_in * size + n_out * 4), "flops": 2 * visits * b}
    if what == "literal":
        return {"bytes": brain + b * n * 8, "flops": 2 * synapses * (case["steps"] - 1) * b}
    moves = 32 * (8 + 8 + 4) if what == "evaluator" and not case["lazy"] else N_MOVES * (2 if what == "evaluator" else 4)
    io = b * (k * size + moves + 12)
    if what == "train":
        return {"bytes": 2 * (brain + 4 * dense) + io, "flops": 3 * 2 * (visits + dense) * b}
    return {"bytes": brain + 4 * dense + io, "flops": 2 * (visits + dense) * b}


# About four times what the path shows against float64 over the ranges above: in relative 2-norm and largest difference.
# The half-precision state's rounding (1.2e-4, 1.6e-3 at one value) grows in the heads, the softmax and the half-precision
# answers (3.5e-4, 1.3e-3).  The float32 sums show 8e-8 and 1.1e-6, with the dense maps 6e-7 and 4e-6.  A gradient
# shows 2e-6 and 7e-4, and up to 2e-5 where a drive lies within rounding of a clamp's bound, which lets a whole column
# of its neuron's gradient through or not.
TOLERANCE = {"model f16": (1e-3, 5e-3), "model f32": (2.5e-6, 2e-5), "io f16": (5e-4, 7e-3), "io f32": (5e-7, 5e-6),
             "literal f32": (5e-7, 5e-6), "evaluator f16": (1.5e-3, 6e-3), "train f32": (1e-4, 0.1),
             "refresh f16": (1e-3, 5e-3)}


def tolerance(case):
    rel, most = TOLERANCE[case["what"] + " " + case["dtype"]]
    return {"rel": rel, "max": most}


# ---- the same in float64, by torch alone ----------------------------------------------------------------------------

class _Product64(torch.autograd.Function):
    """y = A h in float64 for the CSR matrix of edge weights w, with both gradients."""

    @staticmethod
    def forward(ctx, h, w, g):
        ctx.save_for_backward(h, w)
        ctx.g = g
        return torch.sparse_csr_tensor(g["crow"], g["pre"], w, (g["n"], g["n"])) @ h

    @staticmethod
    def backward(ctx, gy):
        h, w = ctx.saved_tensors
        g = ctx.g
        at = torch.sparse_csr_tensor(g["t_crow"], g["post"][g["t_order"]], w[g["t_order"]], (g["n"], g["n"]))
        gy = gy.contiguous()
        gw = torch.empty_like(w)
        for i in range(0, w.numel(), 1 << 18):
            s = slice(i, i + (1 << 18))
            gw[s] = (gy[g["post"][s]] * h[g["pre"][s]]).sum(1)
        return at @ gy, gw, None


def _arrays64(kind, state):
    """The graph's arrays and the float64 widening of a state dict."""
    conn, scale = _graph(kind)
    n = conn.n_neurons
    pre, post = conn.pre.to(DEV), conn.post.to(DEV)
    order = torch.argsort(pre * n + post)

    def crow(rows):
        c = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        c[1:] = torch.bincount(rows, minlength=n).cumsum(0)
        return c

    g = {"n": n, "pre": pre, "post": post, "crow": crow(post), "t_crow": crow(pre), "t_order": order,
         "in": conn.nodes("afferent").to(DEV), "out": conn.nodes("efferent").to(DEV),
         "w0": (conn.weight * scale).to(DEV).double() * conn.sign.to(DEV).double()}
    return g, {k: v.double() for k, v in state.items()}


def _recur64(g, p, u, steps):
    """The state of every neuron after `steps` updates under the constant drive u (n, batch)."""
    w = g["w0"] * torch.exp(p["brain.log_gain"])
    alpha = torch.sigmoid(p["brain.alpha_logit"]).unsqueeze(1)
    drive = u + p["brain.bias"].unsqueeze(1)
    h = alpha * drive.clamp(0, 10)
    for _ in range(steps - 1):
        h = torch.lerp(h, (_Product64.apply(h, w, g) + drive).clamp(0, 10), alpha)
    return h


def _model64(case, g, p, x, u=None, batch_norm=False):
    if u is None:
        k = N_FEATURES if case["planes"] else N_BASE
        u = (F.linear(x[:, :k].double(), p["encoder.weight"][:, :k], p["encoder.bias"]) * GAIN).T
    full = torch.zeros(g["n"], u.shape[1], dtype=torch.float64, device=DEV).index_copy(0, g["in"], u)
    r = _recur64(g, p, full, case["steps"])[g["out"]]
    if case["what"] == "io":
        return r
    r = r.T
    mean, var = (r.detach().mean(0), r.detach().var(0)) if batch_norm else (p["norm.mean"], p["norm.var"])
    r = ((r - mean) / (var + 1e-8).sqrt()).clamp(-8, 8)
    frm, to = (torch.as_tensor(a, device=DEV) for a in move_squares())
    head = lambda name: F.linear(r, p[name + ".weight"], p[name + ".bias"])  # noqa: E731
    return head("policy") + head("policy_from")[:, frm] + head("policy_to")[:, to], head("value")


def exact(case, seed):
    what = case["what"]
    key = (case["graph"], case["steps"], case["planes"], case["dtype"])
    if what == "train":
        net = _net(*key, "train")
        state = {k: v.detach() for k, v in net.state_dict().items()}
        g, p = _arrays64(case["graph"], state)
        params = [k for k, _ in net.named_parameters()]
        for k in params:
            p[k].requires_grad_(True)
        with torch.no_grad():
            x, (pi, legal, wdl) = _boards(case, seed), _targets(case, seed)
        logits, value = _model64(case, g, p, x, batch_norm=True)
        loss = _loss(logits, value, pi.double(), legal, wdl)
        loss.backward()
        return {"loss": loss.detach(), "logits": logits.detach(), "wdl": value.detach(),
                "grads": {k: p[k].grad for k in params}}
    with torch.no_grad():
        x = _boards(case, seed)
        net = _template(case["graph"])
        state = _draw_weights(net, seed) if what == "refresh" else net.state_dict()
        g, p = _arrays64(case["graph"], state)
        if what == "literal":
            u = torch.zeros(g["n"], case["batch"], dtype=torch.float64, device=DEV)
            u[g["in"]] = _drive(net, x, torch.float32).double()
            return _recur64(g, p, u, case["steps"])
        parts = []
        for i in range(0, case["batch"], 512):                           # positions are independent of each other
            xs = x[i:i + 512]
            u = _drive(net, xs, DTYPES[case["dtype"]]).double() if what == "io" else None
            parts.append(_model64(case, g, p, xs, u))
        if what == "io":
            return torch.cat(parts, 1)
        logits, value = (torch.cat(v) for v in zip(*parts))
        if what != "evaluator":
            return logits, value
        rows, cols = (None, None) if case["lazy"] else _legal(case, seed)
        q = value.softmax(-1)
        return (logits if case["lazy"] else logits[rows, cols]).cpu().numpy(), (q[:, 0] - q[:, 2]).cpu().numpy()
