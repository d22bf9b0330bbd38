"""The calls whose speed this repository answers for.

Each case is one use of the package through its public entry points, at the
sizes of the models it serves (hidden 512 / 1024 / 3072 / 4096: the proxy, 1B,
3B and 8B models, with 28 or 32 layers in up to 8 blocks) or at generic ones
(hidden 768, 1000, 1280, 2048, ...), from one decoded token to a prefill of
32768.  The kinds of call:

``router``     the arena loop over every routing point of a model (decode and
               prefill); the sublayers' outputs are given
``route``      one routing point over a padded buffer (``route_static``)
``list``       one routing point over separate blocks
               (``block_attn_res_from_list``)
``weights``    a routing point with the depth-softmax weights
               (``route_weights``, what the monitors read)
``route_grad`` / ``list_grad``  a routing point forward and backward
``loop_grad``  the training loop (``forward_attn_res`` under autograd) of a
               small model, with every gradient
``phase1``     Q pseudo-queries over the committed blocks (serving)
``merge``      the phase-2 merge of the running block into a phase-1 row
``two_phase_grad``  phase 1 and one merge, forward and backward
"""

from __future__ import annotations

import math

import torch

import kotodama_amd
from kotodama_amd.flash_attn_res.ops.phase_1 import phase_1_batched_attention
from kotodama_amd.flash_attn_res.ops.phase_2 import phase_2_online_softmax_merge
from kotodama_amd.schedule import AttnResSchedule

DEVICE = "cuda"
EPS = 1e-5
BF16, FP32 = "bfloat16", "float32"


# ----------------------------------------------------------------- cases --


def listed() -> list:
    return [
        # One sequence decoding one token on the 1B model: 57 tiny calls, all latency.
        dict(name="decode_1b_one_token", kind="router", hidden=1024, batch=1, seq=1, layers=28, blocks=6, dtype=BF16),
        # A full serving batch decoding one token each on the 8B model.
        dict(name="decode_8b_batch256", kind="router", hidden=4096, batch=256, seq=1, layers=32, blocks=8, dtype=BF16),
        # One user's prompt of ragged length prefilled on the 1B model.
        dict(name="prefill_1b_prompt", kind="router", hidden=1024, batch=1, seq=1501, layers=28, blocks=6, dtype=BF16),
        # A routing point of the 3B model's evaluation forward, the deepest one: the largest call.
        dict(name="route_3b", kind="route", hidden=3072, batch=8, seq=4096, sources=8, dtype=BF16),
        # The monitors' weights of a mid-depth point, at a generic width and a ragged row count.
        dict(name="weights_768", kind="weights", hidden=768, batch=5, seq=1637, sources=5, dtype=BF16),
        # An fp32 evaluation through the list form, at a width and a row count that no tile divides.
        dict(name="list_fp32_odd", kind="list", hidden=1000, batch=3, seq=677, sources=4, dtype=FP32),
        # A routing point of a hidden-2048 model's training step, forward and backward.
        dict(name="route_grad_2048", kind="route_grad", hidden=2048, batch=4, seq=2048, sources=5, dtype=BF16),
        # The 8B model's deepest point over separate blocks, forward and backward.
        dict(name="list_grad_8b", kind="list_grad", hidden=4096, batch=2, seq=4096, sources=9, dtype=BF16),
        # The training loop at the proxy model's width and micro-batch, eight layers in four blocks.
        dict(name="loop_grad_proxy", kind="loop_grad", hidden=512, batch=4, seq=2048, layers=8, blocks=4, dtype=BF16),
        # A block of eight sublayers of the 3B model in the two-phase serving forward.
        dict(name="phase1_3b", kind="phase1", hidden=3072, batch=4, seq=4096, sources=4, queries=8, dtype=BF16),
        # The merge of the running block that follows at each of those sublayers.
        dict(name="merge_3b", kind="merge", hidden=3072, batch=4, seq=4096, dtype=BF16),
        # The two phases differentiated at the 1B model's width.
        dict(name="two_phase_grad_1b", kind="two_phase_grad", hidden=1024, batch=4, seq=2048, sources=3, queries=6,
             dtype=BF16),
    ]


WIDTHS = (512, 768, 1000, 1024, 1280, 1536, 2048, 2560, 3072, 3584, 4096)
MODEL_WIDTHS = (512, 1024, 2048, 3072, 4096)


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(("router", "router", "route", "weights", "list", "route_grad", "list_grad", "loop_grad", "phase1",
                       "merge", "two_phase_grad"))
    case = dict(kind=kind, dtype=BF16)
    case["hidden"] = rng.choice(MODEL_WIDTHS if kind == "loop_grad" else WIDTHS)
    if kind == "router":
        decode = rng.random() < 0.5
        case["batch"] = _log_int(rng, 1, 256) if decode else rng.randint(1, 2)
        case["seq"] = 1 if decode else _log_int(rng, 16, 2048)
        case["layers"] = rng.randint(8, 32)
        case["blocks"] = rng.randint(3, 8)
    elif kind == "loop_grad":
        case["batch"] = rng.randint(1, 4)
        case["seq"] = _log_int(rng, 128, 2048)
        case["layers"] = rng.randint(4, 8)
        case["blocks"] = rng.randint(2, 4)
    else:
        case["batch"] = rng.randint(1, 5)
        case["seq"] = _log_int(rng, 64, 4096)
        if kind == "phase1":
            case["sources"] = rng.randint(1, 7)
            case["queries"] = rng.randint(2, 10)
        elif kind == "two_phase_grad":
            case["sources"] = rng.randint(1, 7)
            case["queries"] = rng.randint(2, 8)
        elif kind != "merge":
            case["sources"] = rng.randint(2, 9)
            if kind in ("route", "list", "route_grad") and rng.random() < 0.25:
                case["dtype"] = FP32
    most = max(work(c)["bytes"] for c in listed())
    while work(case)["bytes"] > most:
        case["seq" if case["seq"] > 1 else "batch"] = case["seq" if case["seq"] > 1 else "batch"] * 2 // 3
    return case


# ---------------------------------------------------------------- inputs --


class _Norm:
    """What the routing functions read of a model's RMSNorm."""

    def __init__(self, weight: torch.Tensor) -> None:
        self.weight = weight
        self.eps = EPS


class _Scale(torch.nn.Module):
    """A stand-in sublayer: each feature times a number of its own, one elementwise kernel each way."""

    def __init__(self, factors: torch.Tensor) -> None:
        super().__init__()
        self.register_buffer("factors", factors)

    def forward(self, x, *args):
        return x * self.factors


class _Layer(torch.nn.Module):
    def __init__(self, queries, gains, factors) -> None:
        super().__init__()
        self.attn_norm, self.ffn_norm = torch.nn.Identity(), torch.nn.Identity()
        self.attn, self.ffn = _Scale(factors[0]), _Scale(factors[1])
        self.attn_res_query = torch.nn.Parameter(queries[0].clone())
        self.mlp_res_query = torch.nn.Parameter(queries[1].clone())
        self.attn_res_norm = torch.nn.Module()
        self.mlp_res_norm = torch.nn.Module()
        for norm, gain in ((self.attn_res_norm, gains[0]), (self.mlp_res_norm, gains[1])):
            norm.weight = torch.nn.Parameter(gain.clone())
            norm.eps = EPS


class _Config:
    def __init__(self, layers: int) -> None:
        self.num_layers = layers
        self.norm_eps = EPS


class _Model(torch.nn.Module):
    """The attributes that ``forward_attn_res`` reads of a model."""

    def __init__(self, schedule: AttnResSchedule, queries, gains, factors) -> None:
        super().__init__()
        n = schedule.num_layers
        self.config = _Config(n)
        self.layers = torch.nn.ModuleList(
            [_Layer(*(p[2 * i:2 * i + 2] for p in (queries, gains, factors))) for i in range(n)])
        self.final_res_query = torch.nn.Parameter(queries[-1].clone())
        self.final_res_norm = torch.nn.Module()
        self.final_res_norm.weight = torch.nn.Parameter(gains[-1].clone())
        self.final_res_norm.eps = EPS
        self.norm = torch.nn.Identity()
        self.rope_cos = self.rope_sin = None
        self._attn_res_boundary_set = schedule.boundary_set

    def routing_parameters(self) -> list:
        """Queries and gains in routing-point order."""
        out = []
        for layer in self.layers:
            out += [layer.attn_res_query, layer.attn_res_norm.weight, layer.mlp_res_query, layer.mlp_res_norm.weight]
        return out + [self.final_res_query, self.final_res_norm.weight]


def _schedule(case) -> AttnResSchedule:
    return AttnResSchedule.build(case["layers"], n_blocks=case["blocks"])


def _inputs(case, seed: int) -> dict:
    """The case's tensors: blocks N(0, 1) at scales spread over [0.5, 4], queries
    N(0, 0.05), gains 1 + N(0, 0.1), sublayer outputs and gradients N(0, 1)."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = getattr(torch, case["dtype"])
    d, shape = case["hidden"], (case["batch"], case["seq"], case["hidden"])

    def normal(*size, scale=1.0, to=dt):
        return torch.randn(size, generator=g, device=DEVICE, dtype=torch.float32).mul_(scale).to(to)

    def params(count):
        return normal(count, d, scale=0.05), normal(count, d, scale=0.1, to=torch.float32).add_(1.0).to(dt)

    def stacked(count):
        scales = torch.exp(torch.rand(count, generator=g, device=DEVICE) * math.log(8.0) + math.log(0.5)).tolist()
        buf = torch.empty((count, *shape), device=DEVICE, dtype=dt)
        for i, scale in enumerate(scales):
            buf[i].copy_(normal(*shape, scale=scale))
        return buf

    kind = case["kind"]
    t: dict = {}
    if kind in ("router", "loop_grad"):
        points = 2 * case["layers"] + 1
        t["embed"] = normal(*shape)
        t["queries"], t["gains"] = params(points)
        if kind == "router":
            t["deltas"] = [normal(*shape) for _ in range(points - 1)]
        else:
            t["factors"], t["grad"] = normal(points - 1, d), normal(*shape)
    elif kind == "merge":
        t["partial"], t["inter"] = normal(*shape, scale=2.0), normal(*shape)
        t["lse"] = normal(*shape[:-1], to=torch.float32)
        t["query"] = normal(d, scale=0.05)
    elif kind == "phase1":
        t["buf"], t["query"] = stacked(case["sources"]), normal(case["queries"], d, scale=0.05)
    elif kind == "two_phase_grad":
        nq = case["queries"]
        t["buf"], t["query"] = stacked(case["sources"]), normal(nq, d, scale=0.05)
        t["partial"] = normal(*shape, scale=2.0)
        t["grad"], t["grad_merged"] = normal(nq, *shape), normal(*shape)
    else:
        t["buf"] = stacked(case["sources"])
        q, gain = params(1)
        t["query"], t["gain"] = q[0], gain[0]
        if kind in ("route_grad", "list_grad"):
            t["grad"] = normal(*shape)
    return t


def prepare(case, seed: int) -> dict:
    t = _inputs(case, seed)
    kind = case["kind"]
    st = dict(t, kind=kind)
    if kind == "router":
        sched = _schedule(case)
        st["router"] = kotodama_amd.AttnResRouter(sched, list(t["queries"]), list(t["gains"]), EPS)
        st["arena"] = st["router"].new_arena(t["embed"].shape[:-1], case["hidden"], t["embed"].dtype, t["embed"].device)
    elif kind == "loop_grad":
        st["model"] = _Model(_schedule(case), t["queries"], t["gains"], t["factors"])
        st["embed"] = t["embed"].requires_grad_()
    elif "gain" in t:
        st["norm"] = _Norm(t["gain"])
        st["mask"] = torch.ones(case["sources"], dtype=torch.bool, device=DEVICE)
        if kind in ("list", "list_grad"):
            # the blocks of a caller's loop are separate allocations
            st["blocks"] = [b.clone() for b in t["buf"]]
            del st["buf"]
        if kind.endswith("_grad"):
            for leaf in [st["query"], st["norm"].weight] + (st["blocks"] if kind == "list_grad" else [st["buf"]]):
                leaf.requires_grad_()
    elif kind == "two_phase_grad":
        for name in ("buf", "query", "partial"):
            st[name].requires_grad_()
    return st


# ---------------------------------------------------------------- passes --


def run(st):
    kind = st["kind"]
    if kind == "router":
        routed, deltas = [], st["deltas"]

        def sublayer(j, h):
            routed.append(h)
            return deltas[j]

        with torch.no_grad():
            routed.append(st["router"].forward(st["embed"], sublayer, arena=st["arena"]))
        # the arena holds the blocks; the rows of at most 63 points beside it (the 8B model's first two,
        # of one and two sources, are left out)
        return routed[-63:] + [st["arena"].buf]
    if kind == "route":
        with torch.no_grad():
            return kotodama_amd.route_static(st["buf"], st["query"], st["norm"], st["mask"], st["buf"].shape[0])
    if kind == "list":
        with torch.no_grad():
            return kotodama_amd.block_attn_res_from_list(st["blocks"], st["query"], st["norm"])
    if kind == "weights":
        with torch.no_grad():
            return kotodama_amd.route_weights(st["buf"], st["buf"].shape[0], st["query"], st["norm"])
    if kind == "route_grad":
        leaves = [st["buf"], st["query"], st["norm"].weight]
        out = kotodama_amd.route_static(st["buf"], st["query"], st["norm"], st["mask"], st["buf"].shape[0])
        return [out.detach(), *torch.autograd.grad(out, leaves, st["grad"])]
    if kind == "list_grad":
        leaves = [*st["blocks"], st["query"], st["norm"].weight]
        out = kotodama_amd.block_attn_res_from_list(st["blocks"], st["query"], st["norm"])
        return [out.detach(), *torch.autograd.grad(out, leaves, st["grad"])]
    if kind == "loop_grad":
        model, embed = st["model"], st["embed"]
        out = kotodama_amd.forward_attn_res(model, embed)
        return [out.detach(), *torch.autograd.grad(out, [embed, *model.routing_parameters()], st["grad"])]
    if kind == "phase1":
        with torch.no_grad():
            return phase_1_batched_attention(st["buf"], st["query"], EPS)
    if kind == "merge":
        with torch.no_grad():
            return phase_2_online_softmax_merge(st["partial"], st["query"], st["inter"], st["lse"], EPS)
    # two_phase_grad
    buf, query, partial = st["buf"], st["query"], st["partial"]
    out, lse = phase_1_batched_attention(buf, query, EPS)
    merged = phase_2_online_softmax_merge(partial, query[-1], out[-1], lse[-1], EPS)
    grads = torch.autograd.grad([out, merged], [buf, query, partial], [st["grad"], st["grad_merged"]])
    return [out.detach(), lse.detach(), merged.detach(), *grads]


# ------------------------------------------------------------------ work --


def work(case) -> dict:
    """Bytes: each input read once and each output written once.  Operations per
    element: 4 for a source's sum of squares and dot product, 2 for its share of
    a weighted sum; the backward about twice that."""
    d, n = case["hidden"], case["batch"] * case["seq"]
    e = 4 if case["dtype"] == FP32 else 2
    row = n * d * e
    kind = case["kind"]
    s = case.get("sources", 0)
    if kind in ("router", "loop_grad"):
        sched = _schedule(case)
        points, total = sched.num_points, sched.total_sources()
        if kind == "router":
            # per point: its sources, the sublayer output, the updated partial and the routed row; the
            # first point starts from the embedding, and a new block's partial is the sublayer output itself
            rows = total + 3 * (points - 1) + 2 - sum(sched.commit_before)
            return {"bytes": rows * row + 2 * points * d * e, "flops": 6 * n * d * total}
        # forward: sources, sublayer output, routed row and partial; backward: sources, output gradient
        # and partial gradient; per block its gradient once; the sublayers read and write a row each way
        rows = 2 * total + 5 * points + sched.max_sources + 4 * (points - 1)
        return {"bytes": rows * row + 4 * points * d * e, "flops": 18 * n * d * total}
    if kind == "phase1":
        nq = case["queries"]
        return {"bytes": (s + nq) * row + 4 * nq * n + nq * d * e, "flops": n * d * s * (2 + 4 * nq)}
    if kind == "merge":
        return {"bytes": 3 * row + 4 * n + d * e, "flops": 8 * n * d}
    if kind == "two_phase_grad":
        nq = case["queries"]
        # forward: blocks, Q rows, partial, merged; backward: blocks, Q + 1 output gradients, partial, the
        # merged query's row, block and partial gradients
        return {"bytes": (s + nq + 2 + s + nq + 1 + 2 + s + 1) * row + 8 * nq * n, "flops": n * d * (s * (4 + 12 * nq) + 24)}
    if kind in ("route_grad", "list_grad"):
        return {"bytes": (s + 1 + 2 * s + 1) * row + 6 * d * e, "flops": 18 * n * d * s}
    extra = 4 * n * (s + 1) if kind == "weights" else 0
    return {"bytes": (s + 1) * row + 2 * d * e + extra, "flops": 6 * n * d * s}


def tolerance(case):
    """Four times the distance from float64 of the same inputs that was measured
    over these ranges: one rounding to bf16 (1.7e-3), or fp32 sums."""
    if case["kind"] == "loop_grad":
        # each routed row and partial sum is rounded to bf16 on its way through the layers
        return {"rel": 0.03, "max": 0.9}
    if case["dtype"] == FP32:
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 8e-3, "max": 0.2}


# ----------------------------------------------------------------- exact --


def _fold(query, gain):
    """query * gain, rounded to the parameters' type as the routing defines it."""
    qw = query.double() * gain.double()
    return qw + ((query.detach() * gain.detach()).double() - qw).detach()


def _mix(sources, qw, want=False):
    """Routing over a list of (..., D) float64 sources."""
    logits = torch.stack([(x @ qw) * torch.rsqrt(x.square().mean(-1) + EPS) for x in sources])
    w = torch.softmax(logits, 0)
    out = sources[0] * w[0].unsqueeze(-1)
    for x, ws in zip(sources[1:], w[1:]):
        out = out + x * ws.unsqueeze(-1)
    return (out, w, torch.logsumexp(logits, 0)) if want else out


def exact(case, seed: int):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "router":
        sched = _schedule(case)
        dt = t["embed"].dtype
        blocks, outs = [t["embed"]], []
        for j in range(sched.num_points):
            if j:
                delta = t["deltas"][j - 1]
                if sched.commit_before[j]:
                    blocks.append(delta)
                else:
                    blocks[-1] = (blocks[-1].double() + delta.double()).to(dt)  # the partial is a tensor of that type
            outs.append(_mix([b.double() for b in blocks], _fold(t["queries"][j], t["gains"][j])))
        return outs[-63:] + [torch.stack([b.double() for b in blocks])]
    if kind == "loop_grad":
        sched = _schedule(case)
        embed = t["embed"].double().requires_grad_()
        queries = [q.double().requires_grad_() for q in t["queries"]]
        gains = [g.double().requires_grad_() for g in t["gains"]]
        blocks, h = [embed], None
        for j in range(sched.num_points):
            if j:
                delta = h * t["factors"][j - 1].double()
                if sched.commit_before[j]:
                    blocks = blocks + [delta]
                else:
                    blocks = blocks[:-1] + [blocks[-1] + delta]
            qw = queries[j] * gains[j]
            qw = qw + ((t["queries"][j] * t["gains"][j]).double() - qw).detach()
            h = _mix(blocks, qw)
        leaves = [embed]
        for q, g in zip(queries, gains):
            leaves += [q, g]
        return [h.detach(), *torch.autograd.grad(h, leaves, t["grad"].double())]
    if kind == "merge":
        p, q, inter = t["partial"].double(), t["query"].double(), t["inter"].double()
        return _merge(p, q, inter, t["lse"].double())
    if kind in ("phase1", "two_phase_grad"):
        grad = kind == "two_phase_grad"
        buf = t["buf"].double().requires_grad_(grad)
        query = t["query"].double().requires_grad_(grad)
        res = [_mix(list(buf), q, want=True) for q in query]
        out, lse = torch.stack([r[0] for r in res]), torch.stack([r[2] for r in res])
        if not grad:
            return out, lse
        partial = t["partial"].double().requires_grad_()
        merged = _merge(partial, query[-1], out[-1], lse[-1])
        grads = torch.autograd.grad([out, merged], [buf, query, partial], [t["grad"].double(), t["grad_merged"].double()])
        return [out.detach(), lse.detach(), merged.detach(), *grads]
    if not kind.endswith("_grad"):
        qw = _fold(t["query"], t["gain"])
        rows = [_mix([x.double() for x in t["buf"][:, b]], qw, want=True) for b in range(case["batch"])]
        out, w, lse = (torch.stack([r[i] for r in rows], 1 if i == 1 else 0) for i in range(3))
        return (out, w, lse) if kind == "weights" else out
    buf = t["buf"].double().requires_grad_()
    query, gain = t["query"].double().requires_grad_(), t["gain"].double().requires_grad_()
    qw = query * gain
    out = _mix(list(buf), qw + ((t["query"] * t["gain"]).double() - qw).detach())
    grads = torch.autograd.grad(out, [buf, query, gain], t["grad"].double())
    if kind == "list_grad":
        grads = [*grads[0], grads[1], grads[2]]
    return [out.detach(), *grads]


def _merge(partial, query, inter, lse):
    logit = (partial @ query) * torch.rsqrt(partial.square().mean(-1) + EPS)
    return inter + torch.sigmoid(logit - lse).unsqueeze(-1) * (partial - inter)
