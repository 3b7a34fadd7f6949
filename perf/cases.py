"""The work that programs using flashlog_amd have it do, as measurable cases.

A case is a dict of plain values.  Its ``family`` says which public entry
points one pass goes through:

  sparse    one hop of the models' --sparse path on a coalesced COO state
            [batch, channels, entities]: the hop (all edges, or with the c1
            entity and c2 edge budgets; sum or max), normalize_sparse3d and, in
            training, the backward to state, attention and edge weights;
  channel   the channel reduction after the last hop, with its backward;
  dense     one hop of the dense models: CSR-ordered masks, c1, the sum or max
            hop and, in training, the backward;
  rank      filtered ranks of an evaluation batch, dense or COO scores;
  rules     rule-bank scoring, one score() call per head relation;
  ground    the soft-grounding walk sampler on a batch of head relations.

Graphs follow the laws of the repository's benchmark configurations (uniform
or Zipf relations and degrees); states are drawn as the endpoints of random
triples, so that popular entities are in many rows, valued by how often they
were drawn times a log-normal factor and normalized per row, as the hops
leave them; attention rows are a softmax of N(0, 1) logits.
"""
import functools
import json
import math

import numpy as np
import torch

from flashlog_amd.flashlog_kernel import flashlog_kernel as fk
from flashlog_amd.flashlog_kernel.soft_grounding_kernel import soft_grounding_kernel as sg
from flashlog_amd.rules import shared_inference

DEV = "cuda"
EPS = 1e-7            # the models' normalization floor
NO_BUDGET = 1 << 60   # topk_edges of a hop without an edge budget
LENGTH_CAPS = (64, 4096, 16384)  # the extraction's candidates per head and body length

# (entities, relations, triples, relation law, degree law) of the benchmark
# configurations: small uniform, medium, many-relation, large, web-scale
SMALL = (3_000, 12, 28_000, 0.0, 0.0)
MEDIUM = (41_000, 11, 87_000, 0.0, 1.1)
RELATIONAL = (14_500, 237, 272_000, 1.0, 1.1)
LARGE = (123_000, 37, 1_080_000, 0.0, 1.2)
WEB = (4_600_000, 822, 20_000_000, 1.0, 1.3)


def _graph(g):
    return dict(zip(("entities", "relations", "triples", "rel_law", "deg_law"), g))


def _sparse(g, batch, draws, op="sum", train=False, c1=0, c2=0, channels=3, soft=False, neural=False):
    return dict(family="sparse", **_graph(g), batch=batch, channels=channels, draws=draws, op=op, train=train, c1=c1,
                c2=c2, soft=soft, neural=neural)


def _dense(g, batch, draws, op="sum", train=False, c1=0, c2=0, channels=3, neural=False):
    return dict(family="dense", **_graph(g), batch=batch, channels=channels, draws=draws, op=op, train=train, c1=c1,
                c2=c2, neural=neural)


def listed():
    def named(name, case):
        return dict(case, name=name)

    return [
        # the first hop of a handful of queries from their one-hot states on a small graph, as a
        # program that answers single requests makes it: launches and host work
        named("hop small request", _sparse(SMALL, 4, 1)),
        # training with trainable edge weights and no budgets on a small graph: every edge, each
        # item's gradient also to its edge weight
        named("hop small train edge weights", _sparse(SMALL, 32, 700, train=True, soft=True)),
        # the ordinary training hop: sampled entity and edge budgets on a medium graph
        named("hop medium train", _sparse(MEDIUM, 32, 8_000, train=True, c1=1000, c2=400)),
        # the max models' (mmDRUM) training hop on a large graph
        named("hop large max train", _sparse(LARGE, 32, 10_000, op="max", train=True, c1=1000, c2=400)),
        # the largest training hop: the last one of a web-scale batch
        named("hop web train", _sparse(WEB, 256, 40_000, train=True, c1=1000, c2=400)),
        # the same hop in an evaluation batch: deterministic budgets, no gradients
        named("hop web eval", _sparse(WEB, 256, 40_000, c1=1000, c2=400)),
        # the channel sum of a web-scale batch's last state and its backward
        named("channel sum web", dict(family="channel", **_graph(WEB), batch=256, channels=3, draws=200_000, op="sum",
                                      train=True)),
        # the dense model's training hop on a medium graph
        named("dense medium train", _dense(MEDIUM, 32, 8_000, train=True, c1=1000, c2=400)),
        # the dense max model's training hop on a large graph
        named("dense large max train", _dense(LARGE, 32, 10_000, op="max", train=True, c1=1000, c2=400)),
        # filtered ranking of an evaluation batch over all entities of a large graph
        named("rank large", dict(family="rank", entities=LARGE[0], batch=509, fill=0.3, known=40, dense=True,
                                 ties=True)),
        # rule-bank scoring of some head relations of a rule bank, one call each
        named("rules relational", dict(family="rules", **_graph(RELATIONAL), heads=24, queries=10, rules=42, ranks=3,
                                       op="sum", chunk=64)),
        # soft grounding with the extraction's defaults: 16 heads, up to 512 sources each
        named("grounding relational", dict(family="ground", **_graph(RELATIONAL), heads=16, sources=512, walks=4096,
                                           topk=200)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draws(rng, hi):
    """One-hot first-hop states one time in six, else states of 8 to hi drawn endpoints."""
    return 1 if rng.random() < 1 / 6 else _log_int(rng, 8, hi)


def draw(rng):
    """One more case of the listed ones' ranges."""
    family = rng.choice(["sparse", "sparse", "sparse", "sparse", "dense", "dense", "channel", "rank", "rules", "ground"])
    if family == "rank":
        return dict(family="rank", entities=_log_int(rng, 3_000, 123_000), batch=_log_int(rng, 1, 512),
                    fill=rng.uniform(0.05, 0.9), known=rng.randint(0, 60), dense=rng.random() < 0.5,
                    ties=rng.random() < 0.5)
    if family in ("rules", "ground"):
        relations = _log_int(rng, 11, 237)
        entities = _log_int(rng, 3_000, 14_500)
        g = (entities, relations, rng.randint(3 * entities, 18 * entities), rng.choice([0.0, 1.0]),
             rng.choice([0.0, 1.1]))
        if family == "rules":
            return dict(family="rules", **_graph(g), heads=rng.randint(1, 16), queries=rng.randint(1, 12),
                        rules=rng.randint(1, 60), ranks=rng.randint(1, 3), op=rng.choice(["sum", "max"]), chunk=64)
        return dict(family="ground", **_graph(g), heads=rng.randint(1, 12), sources=_log_int(rng, 8, 512),
                    walks=_log_int(rng, 256, 4096), topk=rng.choice([20, 100, 200]))
    train = rng.random() < 0.5
    if family == "dense":
        entities = _log_int(rng, 3_000, 123_000)
        g = (entities, _log_int(rng, 11, 237), rng.randint(2 * entities, 9 * entities), rng.choice([0.0, 1.0]),
             rng.choice([0.0, 1.1, 1.2]))
        neural = rng.random() < 0.25
        budget = entities > 20_000 or rng.random() < 0.6
        return _dense(g, _log_int(rng, 1, 32), _draws(rng, 10_000), rng.choice(["sum", "sum", "max"]), train,
                      rng.randint(300, 1500) if budget else 0, rng.choice([100, 200, 400]) if budget else 0,
                      1 if neural else rng.randint(1, 4), neural)
    entities = _log_int(rng, 3_000, 2_300_000)
    triples = min(12_000_000, rng.randint(2 * entities, 9 * entities))
    rel_law = rng.choice([0.0, 1.0])
    if family == "channel":
        g = (entities, _log_int(rng, 11, 822), triples, rel_law, rng.choice([1.1, 1.2, 1.3]))
        return dict(family="channel", **_graph(g), batch=_log_int(rng, 1, 128), channels=rng.randint(1, 4),
                    draws=_log_int(rng, 100, 100_000), op=rng.choice(["sum", "max"]), train=train)
    batch = _log_int(rng, 1, 128)
    if entities <= 20_000 and rng.random() < 0.5:
        # no budgets: every edge of every entry
        g = (entities, _log_int(rng, 11, 237), rng.randint(2 * entities, 9 * entities), rel_law, 0.0)
        neural = rng.random() < 0.25
        return _sparse(g, min(batch, 32), _draws(rng, 1_000), "sum", train, 0, 0,
                       1 if neural else rng.randint(1, 3), soft=train and rng.random() < 0.4, neural=neural)
    g = (entities, _log_int(rng, 11, 822), triples, rel_law, rng.choice([0.0, 1.1, 1.2, 1.3]))
    op = rng.choice(["sum", "sum", "max"])
    neural = op == "sum" and rng.random() < 0.2
    return _sparse(g, min(batch, 64) if op == "max" else batch, _draws(rng, 20_000), op, train,
                   rng.randint(200, 1200), rng.choice([50, 100, 200, 400]), 1 if neural else rng.randint(1, 4),
                   neural=neural)


# ---------------------------------------------------------------------------
# Inputs

def _generator(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _law(k, s, count, g):
    """count draws from 0..k-1, uniform or Zipf(s) over a random order."""
    if s == 0:
        return torch.randint(0, k, (count,), generator=g, device=DEV)
    p = torch.arange(1, k + 1, device=DEV, dtype=torch.float64) ** -s
    cdf = torch.cumsum(p[torch.randperm(k, generator=g, device=DEV)], 0)
    x = torch.rand(count, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    return torch.searchsorted(cdf, x).clamp_(max=k - 1)


def _triples(case, g):
    M = case["triples"]
    return (_law(case["entities"], case["deg_law"], M, g), _law(case["relations"], case["rel_law"], M, g),
            _law(case["entities"], case["deg_law"], M, g))


def _state(case, h, t, g):
    """(indices [3, nnz], values) of a coalesced normalized state."""
    E, L, draws = case["entities"], case["channels"], case["draws"]
    rows = case["batch"] * L
    pick = torch.randint(0, h.numel(), (rows * draws,), generator=g, device=DEV)
    ends = torch.where(torch.rand(rows * draws, generator=g, device=DEV) < 0.5, h[pick], t[pick])
    row = torch.arange(rows, device=DEV).repeat_interleave(draws)
    keys, counts = torch.unique(row * E + ends, return_counts=True)
    row, ent = keys // E, keys % E
    v = counts.double()
    if draws > 1:
        v = v * torch.exp(torch.randn(keys.numel(), generator=g, device=DEV, dtype=torch.float64))
    v = (v / torch.zeros(rows, device=DEV, dtype=torch.float64).index_add_(0, row, v)[row]).float()
    return torch.stack([row // L, row % L, ent]), v


def _attention(case, g):
    width = 2 * case["relations"] + (0 if case["neural"] else 1)
    return torch.softmax(torch.randn(case["batch"], case["channels"], width, generator=g, device=DEV), -1)


def _inputs(case, seed):
    """The raw inputs of a sparse, channel or dense case, without this repository's code."""
    g = _generator(seed)
    s = {"case": case, "seed": int(seed)}
    s["h"], s["r"], s["t"] = _triples(case, g)
    s["idx"], s["v"] = _state(case, s["h"], s["t"], g)
    s["shape"] = (case["batch"], case["channels"], case["entities"])
    if case["family"] != "channel":
        s["w"] = _attention(case, g)
        s["hidden"] = torch.randint(0, case["triples"], (case["batch"],), generator=g, device=DEV)
    if case["family"] == "dense":
        b, l, e = s["idx"]
        s["A"] = torch.zeros(s["shape"], device=DEV).index_put_((b, l, e), s["v"])
        if case["train"]:
            s["g"] = torch.rand(s["shape"], generator=g, device=DEV)
    elif case["train"]:
        s["u"] = torch.rand(case["entities"], generator=g, device=DEV)  # upstream gradient by entity
    if case.get("soft"):
        s["weight"] = torch.randn(case["triples"], 1, generator=g, device=DEV)
    return s


def _rank_inputs(case, seed):
    g = _generator(seed)
    B, E = case["batch"], case["entities"]
    scores = torch.rand(B, E, generator=g, device=DEV)
    if case["ties"]:
        scores = torch.round(scores * 4096) / 4096  # several paths of equal weight
    scores = scores * (torch.rand(B, E, generator=g, device=DEV) < case["fill"])
    targets = torch.randint(0, E, (B,), generator=g, device=DEV)
    fb = torch.arange(B, device=DEV).repeat_interleave(case["known"])
    fe = torch.randint(0, E, (B * case["known"],), generator=g, device=DEV)
    s = {"case": case, "scores": scores, "targets": targets, "filter": (fb, fe)}
    if not case["dense"]:
        coo = scores.to_sparse()
        s["coo"] = (coo.indices()[0].contiguous(), coo.indices()[1].contiguous(), coo.values())
        key = torch.cat([fb * E + fe, torch.arange(B, device=DEV) * E + targets])
        s["keys"] = torch.unique(key)
    return s


def _rule_inputs(case, seed):
    g = _generator(seed)
    h, r, t = _triples(case, g)
    R = case["relations"]
    rng = np.random.default_rng(int(seed))
    batches = []
    for _ in range(case["heads"]):
        rules = [{"body": tuple(int(x) for x in rng.integers(0, 2 * R, int(rng.integers(1, 4)))),
                  "rank_weights": [float(x) for x in rng.random(case["ranks"], dtype=np.float32)]}
                 for _ in range(case["rules"])]
        batches.append((h[torch.randint(0, h.numel(), (case["queries"],), generator=g, device=DEV)], rules))
    return {"case": case, "h": h, "r": r, "t": t, "batches": batches}


def _ground_inputs(case, seed):
    g = _generator(seed)
    h, r, t = _triples(case, g)
    R, n = case["relations"], case["heads"]
    rng = np.random.default_rng(int(seed))
    heads = [int(x) for x in rng.choice(2 * R, n, replace=False)]
    folds = []
    for hd in heads:
        ends = torch.unique((h if hd < R else t)[r == hd % R])
        order = torch.randperm(ends.numel(), generator=g, device=DEV)[:case["sources"]]
        src = ends[order].sort().values.cpu()
        folds.append([src if src.numel() else torch.zeros(1, dtype=torch.int64)])
    att = torch.softmax(torch.randn(n, 3, 3, 2 * R + 1, generator=g, device=DEV), -1).cpu()
    return {"case": case, "h": h, "r": r, "t": t, "heads": heads, "folds": folds, "att": att,
            "seeds": [int(seed) ^ (hd * 0x9E3779B1) for hd in heads]}


def prepare(case, seed):
    """What a program has in hand before the pass: inputs, and the graph's CSR arrays."""
    if case["family"] == "rank":
        return _rank_inputs(case, seed)
    s = {"rules": _rule_inputs, "ground": _ground_inputs}.get(case["family"], _inputs)(case, seed)
    if case["family"] != "channel":
        s["csr"] = fk.build_csr_structure(s["h"], s["t"], s["r"], case["entities"])
    if case["family"] in ("sparse", "dense"):
        s["mask"] = torch.ones(case["triples"], dtype=torch.bool, device=DEV)
    for leaf in ("v", "w", "A", "weight"):
        # (a row of one entry is normalized away: no gradient reaches one-hot states)
        if case.get("train") and leaf in s and not (leaf == "v" and case["draws"] == 1):
            s[leaf].requires_grad_(True)
    if case["family"] == "ground":
        s["csr"] = tuple(a.cpu() for a in s["csr"])
    for raw in ("h", "r", "t"):
        s.pop(raw, None)
    return s


# ---------------------------------------------------------------------------
# Passes

ROOM = 1 << 22  # entries


def _room(n, bound):
    """Room for n results of a kind that has at most bound: the bound where that is small, else ROOM, else a power
    of two, so that batches of a kind have results of one shape."""
    return bound if bound <= ROOM else max(ROOM, 1 << (n - 1).bit_length())


def _bounds(case):
    """The most entries of results whose number follows the data."""
    E, queries = case["entities"], case.get("batch") or case["heads"] * case.get("queries", 0)
    rows = queries * (case["channels"] if case["family"] == "sparse" else 1)
    bounds = {"indices": rows * E, "values": rows * E}
    if case["family"] in ("sparse", "channel"):
        bounds["grad_state"] = case["batch"] * case["channels"] * min(E, case["draws"])
    if case["family"] == "ground":
        bounds["candidates"] = case["heads"] * sum(LENGTH_CAPS)
    return bounds


def _kept(s, **results):
    """The results in the program's own buffers (zero past the end)."""
    held = s.setdefault("held", {})
    bounds = _bounds(s["case"])
    for name, x in results.items():
        room = _room(x.shape[-1], bounds[name])
        if name not in held or held[name].shape[-1] != room:
            held[name] = torch.zeros(*x.shape[:-1], room, dtype=x.dtype, device=x.device)
        held[name][..., :x.shape[-1]].copy_(x)
    return {name: held[name] for name in results}


def _run_sparse(s):
    case, csr, mask, w = s["case"], s["csr"], s["mask"], s["w"]
    R, c1, K = case["relations"], case["c1"], case["c2"] // 2
    budget = case["c2"] > 0
    if case["train"]:
        torch.manual_seed(s["seed"])  # the sampled selections draw from torch's generators
        mask[s["hidden"]] = False     # the batch's triples are hidden for the step
    state = torch.sparse_coo_tensor(s["idx"], s["v"], s["shape"], is_coalesced=True)
    weight = s.get("weight")
    with torch.set_grad_enabled(case["train"]):
        if case["train"] and budget:
            out = fk.normalize_sparse3d(fk.sampled_sparse_propagation(
                state, w, csr, mask, R, weight, case["neural"], c1, K, case["op"]), EPS)
        elif case["op"] == "max":
            B, L, E = s["shape"]
            out = fk.normalize_sparse3d(fk.FlashLogFunctionSparse3DTopKMax.apply(
                *state.indices(), state.values(), w, *csr, mask, weight, B, L, E, R, case["neural"], K, False, c1,
                False), EPS)
        else:
            out = fk.vectorized_operation_sparse3d_csr_sum_norm(
                state, w, csr, mask, R, weight=weight, wot_i=case["neural"], use_topk=budget, topk_edges=K, eps=EPS,
                topk_nodes=c1 if budget else None)
        idx, values = out.indices(), out.values()
        if not case["train"]:
            return _kept(s, indices=idx, values=values)
        leaves = {"grad_state": s["v"], "grad_attention": w, "grad_weight": weight}
        leaves = {k: x for k, x in leaves.items() if x is not None and x.requires_grad}
        grads = dict(zip(leaves, torch.autograd.grad(values, list(leaves.values()), s["u"][idx[2]])))
        mask[s["hidden"]] = True
    if "grad_state" in grads:
        grads.update(_kept(s, grad_state=grads["grad_state"]))
    return {**_kept(s, indices=idx, values=values.detach()), **grads}


def _run_channel(s):
    case = s["case"]
    state = torch.sparse_coo_tensor(s["idx"], s["v"], s["shape"], is_coalesced=True)
    reduce = fk.sum_sp_3d if case["op"] == "sum" else fk.max_sp_3d
    with torch.set_grad_enabled(case["train"]):
        out = reduce(state)
        idx, values = out.indices(), out.values()
        if not case["train"]:
            return _kept(s, indices=idx, values=values)
        grad, = torch.autograd.grad(values, [s["v"]], s["u"][idx[1]])
    return _kept(s, indices=idx, values=values.detach(), grad_state=grad)


def _run_dense(s):
    case, csr, mask = s["case"], s["csr"], s["mask"]
    budget = case["c2"] > 0
    hop = fk.dense_csr_sum_cuda if case["op"] == "sum" else fk.dense_csr_max
    if case["train"]:
        mask[s["hidden"]] = False
    with torch.set_grad_enabled(case["train"]):
        masks = fk.prepare_csr_masks(csr, mask)
        outs = hop(s["A"], s["w"], csr, mask, case["relations"], wot_i=case["neural"], use_topk=budget,
                   topk_nodes=case["c1"], topk_edges=case["c2"] // 2, prepared_masks=masks)
        result = {"identity": outs[0], "forward": outs[1], "inverse": outs[2]}
        if case["train"]:
            grads = torch.autograd.grad(outs, [s["A"], s["w"]], [s["g"]] * 3)
            result = {k: o.detach() for k, o in result.items()}
            result.update(zip(("grad_state", "grad_attention"), grads))
            mask[s["hidden"]] = True
    return result


def _run_rank(s):
    if s["case"]["dense"]:
        return fk.dense_filtered_ranks_cuda(s["scores"], s["targets"], s["filter"], s["case"]["ties"])
    B, E = s["scores"].shape
    return fk.sparse2d_filtered_ranks_cuda(*s["coo"], s["targets"], s["keys"], B, E, s["case"]["ties"])


def _run_rules(s):
    case = s["case"]
    out = [shared_inference.score(None, sources, rules, s["csr"], case["relations"], case["entities"], case["chunk"],
                                  reduction=case["op"]) for sources, rules in s["batches"]]
    return {"sizes": np.array([x._nnz() for x in out]),
            **_kept(s, indices=torch.cat([x.indices() for x in out], 1), values=torch.cat([x.values() for x in out]))}


def _run_ground(s):
    case = s["case"]
    candidates, raw, _ = sg.ground_head_batch_source_folds_sampled_capped_counts(
        s["att"], s["heads"], case["relations"], s["folds"], s["csr"], case["walks"], case["topk"], False, s["seeds"],
        500_000, 16, list(LENGTH_CAPS))
    return {"sizes": np.array([x.shape[0] for x in candidates]), "raw": np.array(raw),
            **_kept(s, candidates=torch.cat(candidates).t())}


def run(state):
    return {"sparse": _run_sparse, "channel": _run_channel, "dense": _run_dense, "rank": _run_rank,
            "rules": _run_rules, "ground": _run_ground}[state["case"]["family"]](state)


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch

def _padded(case, **results):
    bounds = _bounds(case)
    return {k: torch.nn.functional.pad(x, (0, _room(x.shape[-1], bounds[k]) - x.shape[-1]))
            for k, x in results.items()}


def _s64(x):
    return x - (1 << 64) if x >= 1 << 63 else x


def _shr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def _phase(seed, b, l, src, inverse):
    """The rounding phase in [0, 1) of the training quotas: one SplitMix64 output per (b, l, source, side)."""
    z = (b * _s64(0x9E3779B97F4A7C15)) ^ (l * _s64(0xBF58476D1CE4E5B9)) ^ (src * _s64(0x94D049BB133111EB))
    z = z ^ seed ^ _s64(0xD1B54A32D192ED03 if inverse else 0x8CB92BAA3F3D8DD7)
    z = z + _s64(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _s64(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _s64(0x94D049BB133111EB)
    return _shr(z ^ _shr(z, 31), 11).double() * 2.0 ** -53


class _Side:
    """One direction's edges ordered by (source, relation, edge id) and their groups of equal (source, relation)."""

    def __init__(self, src, dst, rel, E, R):
        key = src * R + rel
        self.order = torch.argsort(key, stable=True)
        self.dst = dst[self.order]
        gkey, self.count = torch.unique_consecutive(key[self.order], return_counts=True)
        self.start = torch.cumsum(self.count, 0) - self.count
        self.rel = gkey % R
        self.ptr = torch.searchsorted(gkey, torch.arange(E + 1, device=DEV) * R)


def _segment_cumsum(x, seg, nseg):
    """Inclusive running sums of x within its segments (seg ascending)."""
    c = torch.cumsum(x, 0)
    n = torch.bincount(seg, minlength=nseg)
    first = torch.cumsum(n, 0) - n
    return c - torch.where(first > 0, c[(first - 1).clamp_(min=0)], torch.zeros_like(c[:1]))[seg]


def _takes(side, inverse, b, l, e, wrow, K, seed):
    """(entry, group, kept edges) of every group of the entries e that keeps one: all eligible edges of an entry
    with at most K of them; else the K heaviest (ties in group order) or, with a seed, the training quotas."""
    n = e.numel()
    ng = side.ptr[e + 1] - side.ptr[e]
    ent = torch.repeat_interleave(torch.arange(n, device=DEV), ng)
    grp = torch.arange(ent.numel(), device=DEV) - (torch.cumsum(ng, 0) - ng)[ent] + side.ptr[e][ent]
    if K is None:  # every edge, whatever its weight
        return ent, grp, side.count[grp]
    wv = wrow[ent, side.rel[grp]]
    ok = wv > 0
    ent, grp, wv = ent[ok], grp[ok], wv[ok].double()
    cnt = side.count[grp]
    over = torch.zeros(n, dtype=torch.int64, device=DEV).index_add_(0, ent, cnt) > K
    if not bool(over.any()):
        return ent, grp, cnt
    sel = over[ent]
    oe, ow, oc = ent[sel], wv[sel], cnt[sel]
    if seed is None:
        by = torch.argsort(ow, descending=True, stable=True)
        by = by[torch.argsort(oe[by], stable=True)]
        before = _segment_cumsum(oc[by], oe[by], n) - oc[by]
        kept = torch.empty_like(oc)
        kept[by] = torch.minimum((K - before).clamp_(min=0), oc[by])
    else:
        total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, oe, ow)
        base = torch.minimum(oc, torch.floor(K * ow / total[oe]).long())
        spare = oc - base
        residual = K - torch.zeros(n, dtype=torch.int64, device=DEV).index_add_(0, oe, base)
        spares = torch.zeros(n, dtype=torch.int64, device=DEV).index_add_(0, oe, spare)
        prefix = _segment_cumsum(spare, oe, n)

        def cum(p):
            c = torch.floor(residual[oe].double() * p.double() / spares[oe].double()
                            + _phase(seed, b, l, e, inverse)[oe]).long()
            return torch.where(p == spares[oe], residual[oe], torch.where(p == 0, torch.zeros_like(c), c))

        kept = base + cum(prefix) - cum(prefix - spare)
    cnt = cnt.clone()
    cnt[sel] = kept
    some = cnt > 0
    return ent[some], grp[some], cnt[some]


def _edges(side, ent, grp, take):
    """(entry, position) of the taken edges."""
    rep = torch.repeat_interleave(torch.arange(ent.numel(), device=DEV), take)
    off = torch.arange(rep.numel(), device=DEV) - (torch.cumsum(take, 0) - take)[rep]
    return ent[rep], grp[rep], side.start[grp[rep]] + off


def _c1_kept(row, v, rows, c, noise=None):
    """Indices of the entries kept by the entity budget (row ascending)."""
    nonzero = v != 0
    over = torch.bincount(row[nonzero], minlength=rows) > c
    cand = torch.nonzero(over[row] & nonzero).flatten()
    if not cand.numel():
        return None
    score = v[cand].double()
    if noise is not None:
        score = torch.log(score) - torch.log(noise(cand.numel()))
    by = torch.argsort(score, descending=True, stable=True)
    by = by[torch.argsort(row[cand][by], stable=True)]
    rank = torch.empty_like(cand)
    rank[by] = _segment_cumsum(torch.ones_like(cand), row[cand][by], rows) - 1
    keep = ~over[row]
    keep[cand[rank < c]] = True
    return torch.nonzero(keep).flatten()


def _row_chunks(s, sides, row, e, rows, groups=24_000_000):
    """Row ranges whose entries have about that many groups (and as many edges at most in a handful of rows)."""
    per = sum(x.ptr[e + 1] - x.ptr[e] for x in sides)
    budget = s["case"]["c2"]
    if budget:
        per = per + budget
    else:
        per = per + sum((x.start.new_zeros(1) if not x.count.numel() else
                         torch.cat([torch.cumsum(x.count, 0), x.count.new_zeros(1)])[x.ptr[e + 1] - 1]
                         - torch.cat([x.count.new_zeros(1), torch.cumsum(x.count, 0)])[x.ptr[e]]) for x in sides)
    load = torch.zeros(rows, dtype=torch.int64, device=DEV).index_add_(0, row, per).cpu().tolist()
    lo, total = 0, 0
    for r, x in enumerate(load):
        if r > lo and total + x > groups:
            yield lo, r
            lo, total = r, 0
        total += x
    yield lo, rows


def _sides(s):
    E, R = s["case"]["entities"], s["case"]["relations"]
    return _Side(s["h"], s["t"], s["r"], E, R), _Side(s["t"], s["h"], s["r"], E, R)


def _sparse_exact(case, seed, count=False):
    """run()'s outputs of a sparse case; with count, the sizes its work is told from."""
    s = _inputs(case, seed)
    B, L, E = s["shape"]
    rows, R, train = B * L, case["relations"], case["train"]
    K = case["c2"] // 2 if case["c2"] else None
    if case.get("soft"):
        K = K or NO_BUDGET  # trainable edge weights: the budgeted hop without a budget
    sides = _sides(s)
    bl = s["idx"][0] * L + s["idx"][1]
    sampled = train and case["c2"] > 0
    n_in = bl.numel()
    kept = None
    if case["c2"] and n_in > case["c1"]:
        g = _generator(seed) if sampled else None
        draw_noise = (lambda k: torch.empty(k, dtype=torch.float64, device=DEV).exponential_(generator=g)) if g else None
        kept = _c1_kept(bl, s["v"], rows, case["c1"], draw_noise)
    quota_seed = None
    if sampled:
        quota_seed = int(torch.randint(0, 2 ** 63 - 1, (), generator=torch.Generator().manual_seed(int(seed))))
    pick = kept if kept is not None else torch.arange(n_in, device=DEV)
    row, ent_e, v = bl[pick], s["idx"][2][pick], s["v"][pick].double()
    w = s["w"].reshape(rows, -1)
    w64 = w.double()
    visible = torch.ones(case["triples"], dtype=torch.float64, device=DEV)
    if train:
        visible[s["hidden"]] = 0.0
    factor, slope = visible, None
    if case.get("soft"):
        sig = torch.sigmoid(s["weight"].double().view(-1))
        factor, slope = visible * sig, visible * sig * (1 - sig)
    is_max = case["op"] == "max"
    gv = torch.zeros(n_in, dtype=torch.float64, device=DEV)
    gw = torch.zeros(rows, w.shape[1], dtype=torch.float64, device=DEV)
    ge = torch.zeros(case["triples"], dtype=torch.float64, device=DEV)
    keys_out, vals_out = [], []
    sizes = {"in": n_in, "kept": pick.numel(), "items": 0, "out": 0, "groups": 0, "edges": 0}
    if count:
        src = torch.unique(ent_e)
        sizes["groups"] = int(sum((x.ptr[src + 1] - x.ptr[src]).sum() for x in sides))
        ends = [torch.cat([x.start, x.start.new_full((1,), x.dst.numel())]) for x in sides]
        sizes["edges"] = int(sum((p[x.ptr[src + 1]] - p[x.ptr[src]]).sum() for x, p in zip(sides, ends)))
    for lo, hi in _row_chunks(s, sides, row, ent_e, rows):
        a, z = (int(x) for x in torch.searchsorted(row, torch.tensor([lo, hi], device=DEV)))
        if a == z:
            continue
        r, e, x = row[a:z], ent_e[a:z], v[a:z]
        items = []  # (entry, destination, column, factor, edge id or -1)
        for inverse, side in enumerate(sides):
            wr = w[r, inverse * R:inverse * R + R]
            ent, grp, take = _takes(side, inverse, r // L, r % L, e, wr, K, quota_seed)
            ent, grp, pos = _edges(side, ent, grp, take)
            eid = side.order[pos]
            ok = slice(None)
            if K is not None and not is_max:  # a kept edge that is hidden makes no coordinate
                ok = factor[eid] != 0
            items.append((ent[ok], side.dst[pos[ok]], side.rel[grp[ok]] + inverse * R, factor[eid[ok]], eid[ok]))
            del ent, grp, pos, eid
        if not case["neural"]:
            every = torch.arange(z - a, device=DEV)
            items.append((every, e, torch.full_like(every, w.shape[1] - 1), torch.ones_like(x),
                          torch.full_like(every, -1)))
        ent, dst, col, m, eid = (torch.cat(q) for q in zip(*items))
        del items
        wx = w64[r[ent], col]
        val = x[ent] * wx * m
        keys, slot = torch.unique(r[ent] * E + dst, return_inverse=True)
        sizes["items"] += val.numel()
        sizes["out"] += keys.numel()
        if count:
            continue
        out = torch.zeros(keys.numel(), dtype=torch.float64, device=DEV)
        if is_max:
            out = out.scatter_reduce_(0, slot, val, "amax", include_self=False)
            first = torch.full_like(keys, val.numel()).scatter_reduce_(
                0, slot, torch.where(val == out[slot], torch.arange(val.numel(), device=DEV), val.numel()), "amin")
        else:
            out.index_add_(0, slot, val)
        krow = keys // E
        total = torch.zeros(rows, dtype=torch.float64, device=DEV).index_add_(0, krow, out)
        d = total.clamp(min=EPS)[krow]
        keys_out.append(keys)
        vals_out.append(out / d)
        if not train:
            continue
        up = s["u"].double()[keys % E]
        dot = torch.zeros(rows, dtype=torch.float64, device=DEV).index_add_(0, krow, up * out)
        gs = up / d - torch.where(total >= EPS, dot, torch.zeros_like(dot))[krow] / (d * d)
        gi = gs[slot]
        if is_max:
            gi = gi * (torch.arange(val.numel(), device=DEV) == first[slot])
        gv.index_add_(0, pick[a:z][ent], gi * m * wx)
        gw.view(-1).index_add_(0, r[ent] * w.shape[1] + col, gi * m * x[ent])
        if slope is not None:
            edge = eid >= 0
            ge.index_add_(0, eid[edge], (gi * x[ent] * wx)[edge] * slope[eid[edge]])
    if count:
        return sizes
    keys, vals = torch.cat(keys_out), torch.cat(vals_out)
    result = _padded(case, indices=torch.stack([keys // (E * L), keys // E % L, keys % E]), values=vals)
    if train:
        result["grad_attention"] = gw.view(s["w"].shape)
        if case["draws"] > 1:
            result.update(_padded(case, grad_state=gv))
        if slope is not None:
            result["grad_weight"] = ge.view(s["weight"].shape)
    return result


def _channel_exact(case, seed):
    s = _inputs(case, seed)
    B, L, E = s["shape"]
    keys, slot = torch.unique(s["idx"][0] * E + s["idx"][2], return_inverse=True)
    out = torch.zeros(keys.numel(), dtype=torch.float64, device=DEV)
    v = s["v"].double()
    if case["op"] == "max":
        out.scatter_reduce_(0, slot, v, "amax", include_self=False)
    else:
        out.index_add_(0, slot, v)
    result = _padded(case, indices=torch.stack([keys // E, keys % E]), values=out)
    if case["train"]:
        g = s["u"].double()[keys % E]
        if case["op"] == "max":
            top = (v == out[slot]).double()
            share = torch.zeros_like(out).index_add_(0, slot, top) + (out == 0).double()
            result.update(_padded(case, grad_state=top * (g / share)[slot]))
        else:
            result.update(_padded(case, grad_state=g[slot]))
    return result


def _dense_exact(case, seed):
    s = _inputs(case, seed)
    B, L, E = s["shape"]
    rows, R, train = B * L, case["relations"], case["train"]
    A = s["A"].reshape(rows, E)
    w = s["w"].reshape(rows, -1)
    w64 = w.double()
    row, ent = torch.nonzero(A, as_tuple=True)
    alive = torch.ones(rows, E, dtype=torch.float64, device=DEV)
    if case["c2"] and case["c1"] < E:
        kept = _c1_kept(row, A[row, ent], rows, case["c1"])
        if kept is not None:
            alive[torch.bincount(row, minlength=rows) > case["c1"]] = 0.0
            row, ent = row[kept], ent[kept]
            alive[row, ent] = 1.0
    x = A[row, ent].double()
    visible = torch.ones(case["triples"], dtype=torch.float64, device=DEV)
    if train:
        visible[s["hidden"]] = 0.0
    g = s["g"].reshape(rows, E).double() if train else None
    K = case["c2"] // 2 or NO_BUDGET
    w_id = torch.zeros(rows, 1, dtype=torch.float64, device=DEV) if case["neural"] else w64[:, -1:]
    result = {"identity": (A.double() * alive * w_id).view(s["shape"])}
    gA, gw = torch.zeros(rows, E, dtype=torch.float64, device=DEV), torch.zeros_like(w64)
    if train and not case["neural"]:
        gA += g * w_id
        gw[:, -1] = (g * A.double() * alive).sum(1)
    for inverse, (name, side) in enumerate(zip(("forward", "inverse"), _sides(s))):
        wr = w[row, inverse * R:inverse * R + R]
        i, grp, take = _takes(side, inverse, row // L, row % L, ent, wr, K, None)
        i, grp, pos = _edges(side, i, grp, take)
        m, col = visible[side.order[pos]], side.rel[grp] + inverse * R
        wx = w64[row[i], col]
        val, to = x[i] * wx * m, row[i] * E + side.dst[pos]
        out = torch.zeros(rows * E, dtype=torch.float64, device=DEV)
        if case["op"] == "max":
            out.scatter_reduce_(0, to, val, "amax", include_self=False)
        else:
            out.index_add_(0, to, val)
        result[name] = out.view(s["shape"])
        if train:
            gi = g.reshape(-1)[to] * m
            if case["op"] == "max":
                number = torch.arange(val.numel(), device=DEV)
                first = torch.full((rows * E,), val.numel(), device=DEV).scatter_reduce_(
                    0, to, torch.where(val == out[to], number, val.numel()), "amin")
                gi = gi * (number == first[to])
            gA.view(-1).index_add_(0, row[i] * E + ent[i], gi * wx)
            gw.view(-1).index_add_(0, row[i] * w.shape[1] + col, gi * x[i])
    if train:
        result.update(grad_state=(gA * alive).view(s["shape"]), grad_attention=gw.view(s["w"].shape))
    return result


def _rank_exact(case, seed):
    s = _rank_inputs(case, seed)
    B, E = s["scores"].shape
    open_ = torch.ones(B, E, dtype=torch.bool, device=DEV)
    open_[s["filter"]] = False
    open_[torch.arange(B, device=DEV), s["targets"]] = False
    truth = s["scores"].gather(1, s["targets"][:, None])
    greater = ((s["scores"] > truth) & open_).sum(1).double()
    if not case["ties"]:
        return greater + 1
    return greater + (((s["scores"] == truth) & open_).sum(1).double() + 2) / 2


def _rules_exact(case, seed):
    s = _rule_inputs(case, seed)
    E, R = case["entities"], case["relations"]
    by = torch.argsort(s["r"])
    first = torch.searchsorted(s["r"][by], torch.arange(R + 1, device=DEV)).tolist()
    src, dst = s["h"][by], s["t"][by]
    out = []
    for sources, rules in s["batches"]:
        n = sources.numel()
        start = torch.zeros(n, E, dtype=torch.float64, device=DEV)
        start[torch.arange(n, device=DEV), sources] = 1.0
        scores = torch.zeros(case["ranks"], n, E, dtype=torch.float64, device=DEV)
        for rule in rules:
            x = start
            for op in rule["body"]:
                edge = slice(first[op % R], first[op % R + 1])
                a, b = (src[edge], dst[edge]) if op < R else (dst[edge], src[edge])
                x = torch.zeros_like(x).index_add_(1, b, x[:, a])
                if case["op"] == "max":
                    x = (x > 0).double()
            for k, wk in enumerate(rule["rank_weights"]):
                if case["op"] == "max":
                    torch.maximum(scores[k], wk * x, out=scores[k])
                else:
                    scores[k] += wk * x
        total = (scores / scores.sum(2, keepdim=True).clamp(min=1e-30)).sum(0)
        at = total.nonzero()
        out.append((at.t(), total[at[:, 0], at[:, 1]]))
    return {"sizes": None, **_padded(case, indices=torch.cat([x for x, _ in out], 1), values=torch.cat([x for _, x in out]))}


def exact(case, seed):
    """run()'s outputs in 64 bits; None for the sampler, whose outputs are whole numbers."""
    f = {"sparse": _sparse_exact, "channel": _channel_exact, "dense": _dense_exact, "rank": _rank_exact,
         "rules": _rules_exact}.get(case["family"])
    return f(case, seed) if f else None


# ---------------------------------------------------------------------------
# Work and tolerances

@functools.lru_cache(maxsize=None)
def _sizes(text):
    """Counts of one drawn input of a case (they hardly depend on the seed)."""
    case = json.loads(text)
    if case["family"] == "channel":
        s = _inputs(case, 1)
        key = s["idx"][0] * case["entities"] + s["idx"][2]
        return {"in": key.numel(), "out": int(torch.unique(key).numel())}
    if case["family"] == "dense":
        case = dict(case, soft=False)
    return _sparse_exact(case, 1, count=True)


def work(case):
    """Bytes and operations of one pass: inputs read once, outputs written once, a multiply and an add per kept edge."""
    case = {k: v for k, v in case.items() if k != "name"}
    family, train = case["family"], case.get("train", False)
    if family == "rank":
        cells = case["batch"] * case["entities"] * (1 if case["dense"] else case["fill"])
        return {"bytes": cells * (4 if case["dense"] else 20) + case["batch"] * (12 + 16 * case["known"]),
                "flops": cells}
    if family == "rules":
        # a rule's paths: about degree^2 endpoints of a query reached through its steps, each read and added per rank
        reach = (case["triples"] / case["entities"] / case["relations"]) ** 2 + 4
        paths = case["heads"] * case["queries"] * case["rules"] * reach
        return {"bytes": case["heads"] * case["queries"] * case["entities"] * 4 + 12 * paths,
                "flops": 2 * paths * case["ranks"]}
    if family == "ground":
        # a walk's three steps (an option, an edge) and its record
        walks = case["heads"] * case["sources"] * case["walks"]
        return {"bytes": walks * (3 * 12 + 9), "flops": walks * 3 * 8}
    n = _sizes(json.dumps(case, sort_keys=True))
    if family == "channel":
        return {"bytes": 28 * n["in"] + 20 * n["out"] + (4 * n["out"] + 4 * n["in"] if train else 0),
                "flops": n["in"]}
    width = 2 * case["relations"] + (0 if case["neural"] else 1)
    rows = case["batch"] * case["channels"]
    graph = 10 * n["groups"] + 4 * min(n["edges"], n["items"])
    attention = 4 * rows * width * (2 if train else 1)
    if family == "dense":
        state = 4 * rows * case["entities"]
        moved = state * 4 + attention + graph + (state * 2 if train else 0)
    else:
        moved = 28 * n["in"] + attention + graph + 28 * n["out"] + (4 * n["in"] + 4 * n["out"] if train else 0)
        moved += 8 * case["triples"] if case["soft"] else 0
    return {"bytes": moved, "flops": n["items"] * (6 if train else 2)}


def tolerance(case):
    """About four times the error against 64 bits measured over the ranges: 32-bit sums of a hop's items, added one
    by one (up to 1e4 to a hub), and, after the normalization's backward, differences of such sums; whole numbers
    (coordinates, ranks, walk counts) are the same."""
    family = case["family"]
    if family in ("rank", "ground"):
        return "exact"
    if family == "sparse":
        return {"rel": 2e-4 if case["train"] else 3e-5}
    return {"rel": 6e-6 if family == "dense" else 1e-6}
