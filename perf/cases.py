"""Performance cases of the gradient-sync path: what a program that uses this package has it do, per iteration.

A case is a dict of plain values. Its ``path`` names the entry point:

  engine   ``VSWFlatSync.step``: the whole sync step of a GPU over flat arenas (what the trainer calls)
  hooks    the comm hooks of the K VSWs of a GPU, bucket by bucket, through ``LocalBucketSync``
  bucket   ``sync.sync_bucket``: one bucket handed over by value
  shard    ``ShardSGD`` / ``ShardAdam`` / ``ShardAdamW``.step(): the optimizer alone, one span per tensor
  gram     ``sync.gram``: worker x worker products as a pass of their own (up to sixteen workers)

``listed()`` holds the fixed cases, ``draw(rng)`` makes another one of the same ranges, ``prepare`` builds what the
program holds before the call, ``run`` is one pass, ``work`` the bytes and operations one pass cannot do without,
``tolerance`` how far another correct implementation at the same precision may differ and ``exact`` the same pass in
64-bit arithmetic.
"""
import math
import random

import torch

from jabas_amd import ddp_comm_hooks as H
from jabas_amd import optim, sync
from jabas_amd import workloads as W
from jabas_amd.engine import VSWFlatSync
from jabas_amd.layout import FlatLayout
from jabas_amd.local_sync import LocalBucketSync

DEVICE = "cuda"


def _case(path, **kw):
    case = dict(path=path, model="", elements=0, tensors=0, K=1, grads="fp32", opt="none", stats="none", clip=0.0,
                replicas=0, aggregate=True)
    unknown = set(kw) - set(case) - {"name"}
    if unknown:
        raise KeyError(f"unknown case fields {sorted(unknown)}")
    case.update(kw)
    return case


def listed():
    return [
        # One small bucket handed over by value with its statistics, the first bucket DDP closes (1 MiB cap): the
        # smallest call, launch and argument marshalling.
        _case("bucket", name="bucket_1mib_sgd", elements=300007, tensors=9, K=2, opt="sgd", stats="similarity"),
        # A small model (or the trainable head of a large one) with eight bf16 VSWs and worker x worker statistics:
        # a step whose launches and host work weigh as much as its bytes.
        _case("engine", name="small_model_k8_gram", elements=1200011, tensors=46, K=8, grads="bf16", opt="adamw", stats="gram"),
        # The five benchmark configurations, each the way its training program runs it.
        _case("engine", name="resnet50_sgd", model="resnet50", K=2, opt="sgd"),
        _case("engine", name="faster_rcnn_trainer_sgd", model="faster_rcnn_r50_fpn", K=3, opt="sgd", aggregate=False),
        _case("engine", name="vit_b16_adamw_similarity", model="vit_b16", K=4, opt="adamw", stats="similarity"),
        _case("engine", name="gnmt_adam_clipped", model="gnmt", K=4, opt="adam", clip=5.0),
        _case("engine", name="vit_l16_bf16_similarity", model="vit_l16", K=8, grads="bf16", opt="adamw", stats="similarity"),
        # Sixteen replicas of a small model on one 288 GB GPU, every worker's gradient norm wanted.
        _case("engine", name="resnet50_k16_bf16_full", model="resnet50", K=16, grads="bf16", opt="sgd", stats="full"),
        # Replicas that keep weight storage of their own, refreshed by the step (the reference's copy to the other VSWs).
        _case("engine", name="resnet50_k4_replicas", model="resnet50", K=4, opt="sgd", replicas=3),
        # The comm hooks as DDP calls them on a statistic step: 14 buckets, four VSWs, the update in the hook.
        _case("hooks", name="vit_b16_hooks", model="vit_b16", K=4, opt="adamw", stats="similarity"),
        # The optimizer on its own over 152 parameter tensors, gradients already averaged.
        _case("shard", name="vit_b16_shard_adamw", model="vit_b16", opt="adamw"),
        # Products between more workers than the sync launch carries.
        _case("gram", name="gram_fp32_k12", elements=25557033, K=12),
    ]


# Most bytes a drawn case may need: those of the largest listed one.
_MAX_BYTES = 44 * 304326632


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("engine",) * 5 + ("bucket", "bucket", "hooks", "shard", "gram", "gram"))
    while True:
        grads = rng.choice(("fp32", "fp32", "bf16"))
        opt = rng.choice(("sgd", "adam", "adamw", "adamw", "adamw_amsgrad"))
        if path == "engine":
            K = rng.choice((1, 2, 3, 4, 4, 5, 6, 8, 8, 12, 16))
            stats = rng.choice(("none", "none", "similarity", "full") + (("gram",) if K <= 8 else ()))
            case = _case("engine", elements=_log_uniform(rng, 1 << 16, 300_000_000), tensors=rng.randint(4, 300), K=K,
                         grads=grads, opt=opt, stats=stats, aggregate=rng.random() < 0.6)
            if rng.random() < 0.2:
                case["clip"] = rng.choice((0.5, 5.0))
            elif rng.random() < 0.2 and K > 1:
                case["replicas"] = K - 1
        elif path == "bucket":
            case = _case("bucket", elements=_log_uniform(rng, 1 << 12, 1 << 25), tensors=rng.randint(1, 60),
                         K=rng.choice((1, 2, 3, 4, 8)), grads=grads, opt=rng.choice((opt, "none")),
                         stats=rng.choice(("none", "similarity", "full")))
        elif path == "hooks":
            case = _case("hooks", elements=_log_uniform(rng, 1 << 20, 100_000_000), tensors=rng.randint(8, 200),
                         K=rng.choice((2, 3, 4, 8)), grads=grads, opt=opt, stats=rng.choice(("none", "similarity")))
        elif path == "shard":
            case = _case("shard", elements=_log_uniform(rng, 1 << 16, 100_000_000), tensors=rng.randint(4, 200), opt=opt)
        else:
            case = _case("gram", elements=_log_uniform(rng, 1 << 16, 100_000_000), K=rng.randint(2, 16), grads=grads)
        if path != "gram" and case["elements"] < 256 * case["tensors"]:
            case["tensors"] = max(1, case["elements"] // 256)
        if work(case)["bytes"] <= _MAX_BYTES:
            return case


# ------------------------------------------------------------------------------------------- sizes and hyperparameters
def _specs(case):
    """Parameter tensors of a case: a benchmark configuration's, or a generic list in which half of the tensors are
    small (norms and biases, no weight decay) and the others share the remaining elements unevenly. Odd sizes."""
    if case["model"]:
        return W.config(case["model"]).specs
    n, count = case["elements"], case["tensors"]
    rng = random.Random(1000003 * count + n)
    small = [rng.randint(1, max(1, min(4096, n // (4 * count)))) for _ in range(count // 2)]
    shares = [math.exp(rng.gauss(0.0, 1.0)) for _ in range(count - len(small))]
    left = n - sum(small)
    big = [max(1, int(left * s / sum(shares))) for s in shares]
    big[-1] += left - sum(big)
    specs = [W.ParamSpec(f"w{i}", size, 1) for i, size in enumerate(big)] + \
            [W.ParamSpec(f"b{i}", size, 0) for i, size in enumerate(small)]
    rng.shuffle(specs)
    return specs


def _batches(case):
    if case["model"]:
        cfg = W.config(case["model"])
        if cfg.K == case["K"]:
            return cfg.batches
    return tuple(16 + 8 * (3 * k % 4) for k in range(case["K"]))


def _opt(case):
    kind = case["opt"]
    if kind == "none":
        return None
    if case["model"] and W.config(case["model"]).opt["kind"] == kind:
        return W.config(case["model"]).opt
    if kind == "sgd":
        return dict(kind="sgd", momentum=0.9, dampening=0.0, nesterov=False,
                    groups=[dict(lr=0.05, weight_decay=0.0), dict(lr=0.05, weight_decay=1e-4)])
    return dict(kind="adam" if kind == "adam" else "adamw", betas=(0.9, 0.999), eps=1e-8, amsgrad=kind.endswith("amsgrad"),
                groups=[dict(lr=5e-4, weight_decay=0.0), dict(lr=5e-4, weight_decay=0.05)])


def _grad_dtype(case):
    return torch.bfloat16 if case["grads"] == "bf16" else torch.float32


def _n_state(case):
    return {"none": 0, "sgd": 1, "adam": 2, "adamw": 2, "adamw_amsgrad": 3}[case["opt"]]


def _numel(case):
    return sum(s.numel for s in W.config(case["model"]).specs) if case["model"] else case["elements"]


# ------------------------------------------------------------------------------------------------------------- inputs
class _Fill:
    """Gradients, weights and optimizer state as a training run meets them: the workers' gradients share a component
    (cosine between the halves near 0.5), the moments are those of a run under way."""
    STD, STEP = 1e-3, 100

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(self, n):
        return torch.randn(n, generator=self.gen, device=DEVICE)

    def gradients(self, buffers):
        common = self.randn(buffers[0].numel())
        for b in buffers:
            own = self.randn(b.numel())
            b.copy_(own.add_(common).mul_(0.7 * self.STD))

    def weights(self, p):
        p.copy_(self.randn(p.numel()).mul_(0.05))

    def state(self, case, j, n):
        if case["opt"] == "sgd":
            return self.randn(n).mul_(3.0 * self.STD)
        if j == 0:
            return self.randn(n).mul_(0.4 * self.STD)
        v = torch.rand(n, generator=self.gen, device=DEVICE).add_(0.5).mul_(self.STD * self.STD)
        return v if j == 1 else v.mul_(1.3)


def _engine(case, seed):
    specs, fill = _specs(case), _Fill(seed)
    eng = VSWFlatSync(specs, _batches(case), grad_dtype=_grad_dtype(case), opt=_opt(case), device=DEVICE,
                      n_fanout=case["replicas"], write_aggregate=case["aggregate"], keep_clipped_grads=case["aggregate"])
    fill.gradients(eng.grads)
    if case["model"] == "gnmt":          # the embedding's gradient touches the rows of the words in the batch only
        i = [s.name for s in specs].index(W.GNMT_EMBEDDING)
        rows = torch.rand(W.GNMT_EMBEDDING_ROWS, 1, generator=fill.gen, device=DEVICE) < 0.1
        for k in range(case["K"]):
            eng.grad_view(k, i).view(W.GNMT_EMBEDDING_ROWS, W.GNMT_EMBEDDING_COLS).mul_(rows)
    fill.weights(eng.param)
    for f in eng.fanout:
        f.copy_(eng.param)
    for j in range(eng.n_state):
        eng.set_state(j, fill.state(case, j, eng.layout.total))
    eng.step_count = fill.STEP
    return eng


def _engine_outputs(case, eng):
    out = {"param": eng.param, "replicas": list(eng.fanout)}
    if case["aggregate"]:
        out["aggregate"] = eng.agg
    for j in range(eng.n_state):
        out[f"state{j}"] = eng.moments.way(j) if eng.moments is not None else (eng.state1, eng.state2, eng.state3)[j]
    return out


class _GradBucket:
    """What the hooks read of a DDP ``GradBucket``."""

    def __init__(self, index, tensor, last):
        self._index, self._tensor, self._last = index, tensor, last

    def index(self):
        return self._index

    def buffer(self):
        return self._tensor

    def is_last(self):
        return self._last


def _prepare_hooks(case, seed):
    eng = _engine(case, seed)
    parts, buckets = {}, []
    for b, (off, numel, bounds, _) in enumerate(eng.layout.spans):
        sl = slice(off, off + numel)
        parts[b] = dict(param=eng.param[sl], bounds=bounds, agg_out=None if eng.in_place else eng.agg[sl],
                        **eng.state_of_span(off, numel))
        last = b + 1 == len(eng.layout.spans)
        buckets.append([_GradBucket(b, g[sl], last) for g in eng.grads])
    local = LocalBucketSync(_batches(case), opt=_opt(case), param_buckets=parts, stream=torch.cuda.Stream())
    local.step_count = eng.step_count
    workers = case["K"] + case["K"] % 2
    state = H.GradientSimilarityState(None, workers, None, [], 1 if case["stats"] != "none" else 10 ** 9)
    state.attach_local(local)
    return dict(engine=eng, local=local, state=state, buckets=buckets,
                main_hook=H.similimarity_allreduce_hook(H.subgroup_allreduce_hook),
                peers=[H.VSWPeerState(local, k) for k in range(1, case["K"])])


def _prepare_bucket(case, seed):
    n, fill = case["elements"], _Fill(seed)
    layout = FlatLayout(_specs(case), caps=(1 << 40,))               # one bucket
    s = dict(batches=_batches(case), dtype=_grad_dtype(case), opt=_opt(case), stats=case["stats"], step=fill.STEP)
    s["grads"] = [torch.empty(n, dtype=s["dtype"], device=DEVICE) for _ in range(case["K"])]
    fill.gradients(s["grads"])
    s["aggregate"] = s["grads"][0] if s["dtype"] == torch.float32 else torch.zeros(n, device=DEVICE)
    s["param"], s["state"] = None, []
    if s["opt"] is not None:
        s["param"] = torch.empty(n, device=DEVICE)
        fill.weights(s["param"])
        s["state"] = [fill.state(case, j, n) for j in range(_n_state(case))]
    bounds = layout.buckets[0].bounds if s["opt"] is not None else ()
    s["span"] = sync.SpanSpec(s["grads"], agg_out=s["aggregate"], param=s["param"], bounds=bounds,
                              **{f"state{j + 1}": t for j, t in enumerate(s["state"])})
    s["bounds_dev"] = sync.bounds_to_device(bounds, torch.device(DEVICE, torch.cuda.current_device())) if bounds else None
    s["workspace"] = sync.Workspace.for_span(n, s["dtype"], DEVICE) if case["stats"] != "none" else None
    return s


def _prepare_shard(case, seed):
    """Weights and moments as the allocator places tensors (512-byte lines), the gradients as DDP packs them."""
    specs, fill = _specs(case), _Fill(seed)
    places, total = [], 0
    for spec in specs:
        places.append((total, spec.numel))
        total += -(-spec.numel // 128) * 128
    layout = FlatLayout(specs)
    flat = dict(param=torch.empty(total, device=DEVICE), grads=torch.empty(layout.total, device=DEVICE),
                state=[fill.state(case, j, total) for j in range(_n_state(case))])
    fill.weights(flat["param"])
    fill.gradients([flat["grads"]])
    opt, groups = _opt(case), {}
    names = ("momentum_buffer",) if opt["kind"] == "sgd" else ("exp_avg", "exp_avg_sq", "max_exp_avg_sq")
    params = []
    for i, (spec, (off, n)) in enumerate(zip(specs, places)):
        p = torch.nn.Parameter(flat["param"][off:off + n])
        g0 = layout.param_offset[i]
        p.grad = flat["grads"][g0:g0 + n]
        groups.setdefault(spec.group, []).append(p)
        params.append(p)
    param_groups = [dict(params=ps, lr=opt["groups"][gi]["lr"], weight_decay=opt["groups"][gi]["weight_decay"])
                    for gi, ps in sorted(groups.items())]
    if opt["kind"] == "sgd":
        flat["opt"] = optim.ShardSGD(param_groups, lr=0.05, momentum=opt["momentum"])
    else:
        cls = optim.ShardAdamW if opt["kind"] == "adamw" else optim.ShardAdam
        flat["opt"] = cls(param_groups, betas=opt["betas"], eps=opt["eps"], amsgrad=opt.get("amsgrad", False))
    for p, (off, n) in zip(params, places):
        st = flat["opt"].state[p]
        for name, t in zip(names, flat["state"]):
            st[name] = t[off:off + n]
        if opt["kind"] != "sgd":
            st["step"] = fill.STEP
    return flat


def _prepare_gram(case, seed):
    grads = [torch.empty(case["elements"], dtype=_grad_dtype(case), device=DEVICE) for _ in range(case["K"])]
    _Fill(seed).gradients(grads)
    return dict(grads=grads)


def prepare(case, seed):
    path = case["path"]
    if path == "engine":
        return dict(case=case, engine=_engine(case, seed))
    make = {"hooks": _prepare_hooks, "bucket": _prepare_bucket, "shard": _prepare_shard, "gram": _prepare_gram}[path]
    return dict(make(case, seed), case=case)


# --------------------------------------------------------------------------------------------------------------- pass
def _run_engine(s):
    case, eng = s["case"], s["engine"]
    stats = False if case["stats"] == "none" else case["stats"]
    rows = eng.step(stats=stats, clip_norm=case["clip"] or None)
    out = _engine_outputs(case, eng)
    if rows is not None:
        out["rows"] = rows
    if stats == "gram":
        out["gram"] = eng.gram(rows)
    return out


def _run_hooks(s):
    state, peers = s["state"], s["peers"]
    for per_vsw in s["buckets"]:
        s["main_hook"](state, per_vsw[0])
        for peer, bucket in zip(peers, per_vsw[1:]):
            H.dummy_hook(peer, bucket)
    s["local"].finish_step((torch.cuda.current_stream(),))
    out = _engine_outputs(s["case"], s["engine"])
    out["rows"] = [stats.row for stats in state.grad_placeholder]
    state.grad_placeholder.clear()
    return out


def _run_bucket(s):
    s["step"] += 1
    stats = False if s["stats"] == "none" else s["stats"]
    args = sync.make_step_args(s["batches"], s["dtype"], stats=stats, opt=s["opt"], step=s["step"])
    row = sync.sync_bucket(s["span"], args, workspace=s["workspace"], bounds_dev=s["bounds_dev"])
    return {"aggregate": s["aggregate"], "param": s["param"], "state": s["state"], "row": row}


def _run_shard(s):
    s["opt"].step()
    return {"param": s["param"], "state": s["state"]}


def _run_gram(s):
    return sync.gram(s["grads"])


_RUN = {"engine": _run_engine, "hooks": _run_hooks, "bucket": _run_bucket, "shard": _run_shard, "gram": _run_gram}


def run(state):
    return _RUN[state["case"]["path"]](state)


# --------------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    """Every gradient read once, weights and optimizer state read and written once, the aggregate and the replicas'
    weights written once; multiply-adds of the aggregate, the statistics and the update rule."""
    n, K = _numel(case), case["K"]
    gs = 2 if case["grads"] == "bf16" else 4
    pairs = K * (K + 1) / 2
    if case["path"] == "gram":
        return {"bytes": n * K * gs, "flops": 2 * n * pairs}
    if case["path"] == "shard":
        return {"bytes": n * (4 + 8 + 8 * _n_state(case)), "flops": n * 14}
    per_elem = K * gs + 4 * case["replicas"]
    if case["aggregate"] or case["opt"] == "none":
        per_elem += 4
    flops = 2 * K
    if case["opt"] != "none":
        per_elem += 8 + 8 * _n_state(case)
        flops += 6 if case["opt"] == "sgd" else 14
    flops += {"none": 0, "similarity": 2 * K + 8, "full": 4 * K + 8, "gram": 2 * K + 8 + 2 * pairs}[case["stats"]]
    return {"bytes": n * per_elem, "flops": n * flops}


def tolerance(case):
    """About four times the distance from the same step in 64-bit arithmetic: single-precision aggregates, moments and
    weights 7e-8 (one element at most 4e-7), the halves behind the statistics 6e-8; products of fp32 gradients, and of
    bf16 gradients of up to seven workers, are summed in fp64; of more bf16 workers in short fp32 runs first."""
    if case["path"] == "gram":
        return {"rel": 4e-7, "max": 8e-7} if case["grads"] == "bf16" and case["K"] > 7 else {"rel": 1e-14, "max": 1e-13}
    return {"rel": 4e-7, "max": 2e-6}


# -------------------------------------------------------------------------------------------------------------- exact
def _sums64(case, grads, halves, agg):
    """Statistics row of a span: the four sums of the halves and the aggregate, every worker's norm, every pair's product."""
    row = torch.zeros(40, dtype=torch.float64, device=DEVICE)
    a, b = halves
    row[:4] = torch.stack([(a * b).sum(), (a * a).sum(), (b * b).sum(), (agg * agg).sum()])
    if case["stats"] in ("full", "gram"):
        row[4:4 + len(grads)] = torch.stack([(g * g).sum() for g in grads])
    if case["stats"] == "gram":
        pairs = [(grads[i] * g).sum() for i in range(len(grads)) for g in grads[i + 1:]]
        row[4 + len(grads):4 + len(grads) + len(pairs)] = torch.stack(pairs) if pairs else row[:0]
    return row


def _update64(opt, group, step, g, p, state):
    """One optimizer step on the 64-bit slices p and state, in place."""
    lr, wd = opt["groups"][group]["lr"], opt["groups"][group]["weight_decay"]
    if opt["kind"] == "sgd":
        state[0].mul_(opt["momentum"]).add_(g + wd * p)
        p.sub_(lr * state[0])
        return
    b1, b2 = opt["betas"]
    if opt["kind"] == "adamw":
        p.mul_(1 - lr * wd)
    else:
        g = g + wd * p
    state[0].mul_(b1).add_(g, alpha=1 - b1)
    state[1].mul_(b2).add_(g * g, alpha=1 - b2)
    second = state[1]
    if opt.get("amsgrad", False):
        second = state[2].copy_(torch.maximum(state[2], state[1]))
    denom = second.sqrt().div_(math.sqrt(1 - b2 ** step)).add_(opt["eps"])
    p.sub_(state[0] / denom * (lr / (1 - b1 ** step)))


def _step64(case, spans, grads, agg, param, state):
    """The sync step on 64-bit copies, span by span: the aggregate into agg, the update into param and state.
    Returns the statistics rows. ``spans``: (first element, elements, [(start, group)], ...)."""
    opt, rows, norm2 = _opt(case), [], 0.0
    b = _batches(case)
    half = [[x / (sum(b[h::2]) or 1) for x in b[h::2]] for h in (0, 1)]
    for off, n, *_ in spans:
        g = [t[off:off + n].double() for t in grads]
        agg[off:off + n] = sum(x * (w / sum(b)) for x, w in zip(g, b))
        if case["stats"] != "none" or case["clip"]:
            halves = [sum((x * w for x, w in zip(g[h::2], half[h])), torch.zeros_like(g[0])) for h in (0, 1)]
            rows.append(_sums64(case, g, halves, agg[off:off + n]))
            norm2 += float(rows[-1][3])
    if case["clip"]:
        coef = case["clip"] / (math.sqrt(norm2) + 1e-6)
        for off, n, *_ in spans:
            agg[off:off + n].mul_(min(1.0, coef))
    if opt is not None:
        for off, n, bounds, *_ in spans:
            ends = [start for start, _ in bounds[1:]] + [n]
            for (start, group), end in zip(bounds, ends):
                sl = slice(off + start, off + end)
                _update64(opt, group, _Fill.STEP + 1, agg[sl], param[sl], [t[sl] for t in state])
    return rows


def _exact_arenas(case, eng):
    state = [s.double() for s in (eng.state1, eng.state2, eng.state3)[:eng.n_state]]
    param = eng.param.double()
    agg = eng.agg.double() if eng.agg is not None else torch.zeros_like(param)
    rows = _step64(case, eng.layout.spans, eng.grads, agg, param, state)
    out = {"param": param, "replicas": [param.clone() for _ in eng.fanout]}
    if case["aggregate"]:
        out["aggregate"] = agg
    for j, t in enumerate(state):
        if eng.moments is not None:
            shape = eng.moments.way(j).shape
            t = torch.nn.functional.pad(t, (0, shape.numel() - t.numel())).view(shape)
        out[f"state{j}"] = t
    return out, rows


def _exact_engine(case, s):
    out, rows = _exact_arenas(case, s["engine"])
    if case["stats"] != "none":
        out["rows"] = torch.stack(rows)
    if case["stats"] == "gram":
        out["gram"] = _gram64([torch.cat([g[o:o + n] for o, n, *_ in s["engine"].layout.spans]) for g in s["engine"].grads])
    return out


def _exact_hooks(case, s):
    out, rows = _exact_arenas(case, s["engine"])
    out["rows"] = rows
    return out


def _exact_bucket(case, s):
    param = None if s["param"] is None else s["param"].double()
    state = [t.double() for t in s["state"]]
    agg = torch.zeros(case["elements"], dtype=torch.float64, device=DEVICE)
    bounds = s["span"].bounds or [(0, 0)]
    rows = _step64(case, [(0, case["elements"], bounds)], s["grads"], agg, param, state)
    return {"aggregate": agg, "param": param, "state": state, "row": rows[0] if rows else None}


def _exact_shard(case, s):
    param, state = s["param"].double(), [t.double() for t in s["state"]]
    opt, layout, off = _opt(case), FlatLayout(_specs(case)), 0
    for spec, g0 in zip(_specs(case), layout.param_offset):
        sl = slice(off, off + spec.numel)
        _update64(opt, spec.group, _Fill.STEP + 1, s["grads"][g0:g0 + spec.numel].double(), param[sl], [t[sl] for t in state])
        off += -(-spec.numel // 128) * 128
    return {"param": param, "state": state}


def _gram64(grads):
    out = torch.zeros(len(grads), len(grads), dtype=torch.float64, device=DEVICE)
    for a, x in enumerate(grads):
        x = x.double()
        for b in range(a + 1):
            out[a, b] = out[b, a] = (x * grads[b].double()).sum()
    return out


def _exact_gram(case, s):
    return _gram64(s["grads"])


_EXACT = {"engine": _exact_engine, "hooks": _exact_hooks, "bucket": _exact_bucket, "shard": _exact_shard, "gram": _exact_gram}


def exact(case, seed):
    """What ``run`` returns for these inputs, in 64-bit torch operations."""
    return _EXACT[case["path"]](case, prepare(case, seed))
