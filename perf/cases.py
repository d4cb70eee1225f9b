"""The workloads this framework's speed is measured on.

Each case is what a user's program has the framework do again and again: a
sampler or optimiser holds a species tree and a set of gene families (their
CCDs, resident on the device) and evaluates the likelihood, or its gradient,
at one parameter point after another.  A pass takes a chain of parameter
points, so every evaluation in it builds the model's tables anew, as a
sampler's does.

Sizes are those of the synthetic workloads (`whale_jl_amd.synth.CONFIGS`) and
of the reference's own examples: 9 to 58 taxa, slices of 0.01 to 0.05 tree
heights, one family to 10,000 families, 4 to 250 genes a family.

Results in FP32 arithmetic carry FP32's digits, so they are returned as
float32; FP64 ones as float64.
"""
import math
import random

import numpy as np
import torch

from __graft_entry__ import load_package

w = load_package()
from whale_jl_amd import synth  # noqa: E402

CONDITIONS = {"root": w.RootCondition, "nonextinct": w.NonExtinctCondition, "none": w.NoCondition}

_DEFAULTS = dict(nwgd=0, ntrees=200, max_clades=100000, mode="fp64", op="gradient", condition="root", points=2,
                 components=1, samples=0, deterministic=False, tree=1)


def _case(**kw):
    return {**_DEFAULTS, **kw}


def listed():
    return [
        # an interactive look at one family: the smallest call there is
        _case(name="one_family_logl", taxa=9, dt=0.05, families=1, median=20, sigma=0.3, lo=8, hi=60, op="logl"),
        # the reference's own benchmark call: 12 families on a 9-taxon tree with 2 WGDs, gradient
        _case(name="dozen_gradient", taxa=9, nwgd=2, dt=0.05, families=12, median=16, sigma=0.3, lo=8, hi=60),
        # the tutorial's size: a hundred families, HMC in the reference's arithmetic
        _case(name="hundred_gradient", taxa=9, dt=0.05, families=100, median=25, sigma=0.6, lo=8, hi=60),
        # one very large family (about 2,000 clades): the batch is one chain of dependent rows
        _case(name="large_family_gradient", taxa=58, dt=0.01, families=1, median=240, sigma=0.03, lo=225, hi=255,
              ntrees=1000),
        # a Metropolis sampler's step in the reference's arithmetic: values only
        _case(name="thousand_logl", taxa=12, nwgd=2, dt=0.02, families=1000, median=30, sigma=0.6, lo=10, hi=150,
              ntrees=500, max_clades=1000, op="logl"),
        # the same families under HMC with the fast form
        _case(name="thousand_gradient_fp32", taxa=12, nwgd=2, dt=0.02, families=1000, median=30, sigma=0.6, lo=10,
              hi=150, ntrees=500, max_clades=1000, mode="fp32"),
        # underflow-free FP64 on a tree of many taxa; bit-identical gradients, as reversible trajectories need;
        # an odd number of families
        _case(name="exact_gradient_fp64s", taxa=50, nwgd=4, dt=0.01, families=777, median=20, sigma=0.9, lo=4, hi=200,
              max_clades=2000, mode="fp64s", deterministic=True),
        # reconciled trees: ℓ at a posterior sample, then trees drawn from it
        _case(name="trees", taxa=13, dt=0.02, families=100, median=30, sigma=0.6, lo=8, hi=120, points=1, samples=4),
        # a mixture of three rate models over the same families, all gradients
        _case(name="mixture_gradient_fp32", taxa=20, nwgd=5, dt=0.02, families=1000, median=25, sigma=0.5, lo=10,
              hi=120, mode="fp32", components=3, points=1),
        # a genome-wide data set on a mid-sized tree under a sampler
        _case(name="sampler_gradient_fp32", taxa=20, nwgd=5, dt=0.02, families=5000, median=25, sigma=0.5, lo=10,
              hi=120, mode="fp32"),
        # values only on the large tree
        _case(name="bulk_logl_fp32", taxa=50, nwgd=4, dt=0.01, families=3001, median=20, sigma=0.9, lo=4, hi=200,
              max_clades=2000, mode="fp32", op="logl"),
        # the headline workload: 10,000 families on 50 taxa and 4 WGDs
        _case(name="bulk_gradient_fp32", taxa=50, nwgd=4, dt=0.01, families=10000, median=20, sigma=0.9, lo=4, hi=200,
              max_clades=2000, mode="fp32"),
    ]


def draw(rng):
    taxa = int(round(math.exp(rng.uniform(math.log(6), math.log(58)))))
    dt = round(math.exp(rng.uniform(math.log(0.01), math.log(0.05))), 4)
    kind = rng.choice(["gradient", "gradient", "gradient", "logl", "logl", "mixture", "trees"])
    c = _case(taxa=taxa, dt=dt, tree=rng.randrange(2, 1000), nwgd=rng.randrange(0, 6), median=rng.randrange(12, 41),
              sigma=round(rng.uniform(0.3, 0.9), 2), lo=rng.choice([4, 6, 8]), hi=rng.choice([80, 120, 150, 200]),
              max_clades=2000, mode=rng.choice(["fp64", "fp32", "fp32", "fp64s"]),
              condition=rng.choice(["root", "root", "nonextinct", "none"]))
    # at most a third of the largest case's families times rows; rows go with taxa / dt
    most = min(5000.0, 10000 * 0.33 * (50 / taxa) * (dt / 0.01))
    c["families"] = int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    if kind == "logl":
        c["op"] = "logl"
    elif kind == "mixture":
        c.update(components=rng.randrange(2, 5), points=1, families=max(1, c["families"] // 4))
    elif kind == "trees":
        c.update(mode="fp64", samples=rng.randrange(1, 5), points=1, families=min(c["families"], 300))
    else:
        c["deterministic"] = rng.random() < 0.2
    return c


# ---------------------------------------------------------------- inputs
_POOLS = {}


def _pool(case):
    """The species tree and the families that cases of this shape draw from
    (a quarter more than a case takes), generated once per process."""
    key = tuple(case[k] for k in ("taxa", "nwgd", "tree", "families", "median", "sigma", "lo", "hi", "ntrees",
                                  "max_clades", "dt"))
    if key not in _POOLS:
        n = case["families"]
        newick = synth.species_tree(1000 + case["tree"], case["taxa"], case["nwgd"])
        texts, _ = synth.families(newick, 77 + case["tree"], n + max(2, n // 4),
                                  ("lognormal", case["median"], case["sigma"], case["lo"], case["hi"]), case["ntrees"],
                                  case["max_clades"], 1000000)
        model = w.WhaleModel(_rates(case, np.random.default_rng(0)), w.readnw(newick), case["dt"])
        _POOLS[key] = newick, list(w.ccds_from_texts(texts, model))
    return _POOLS[key]


def _rates(case, rng):
    n = 2 * case["taxa"] - 1
    lam = math.log(0.2) + 0.5 * rng.standard_normal(n)
    mu = math.log(0.15) + 0.5 * rng.standard_normal(n)
    return w.DLWGD(λ=list(lam), μ=list(mu), q=list(rng.uniform(0.1, 0.6, case["nwgd"])), η=0.9)


def _inputs(case, seed):
    """Newick, families and the chain of parameter points (the components of
    one point, for a mixture) of (case, seed)."""
    newick, pool = _pool(case)
    rng = np.random.default_rng([seed, case["tree"]])
    take = rng.permutation(len(pool))[:case["families"]]
    n = case["components"] if case["components"] > 1 else case["points"]
    points = synth.perturbed(_rates(case, rng), n, seed=int(rng.integers(1 << 30)))
    prior = rng.dirichlet(np.full(case["components"], 5.0)) if case["components"] > 1 else None
    return newick, [pool[i] for i in take], points, prior


def prepare(case, seed):
    newick, fams, points, prior = _inputs(case, seed)
    model = w.WhaleModel(points[0], w.readnw(newick), case["dt"], condition=CONDITIONS[case["condition"]]())
    # CCDs of its own for every state: a CCD keeps its device batch
    ccds = w.CCDSet([w.CCD(c.size, c.leaf_species, c.split_off, c.g1, c.g2, c.p, c.fname) for c in fams])
    one = case["families"] == 1 and case["op"] == "logl"
    if not one:
        batch = w.device_batch(model, ccds)
        if case["deterministic"]:
            batch.set_deterministic(True)
    return {"case": case, "model": model, "ccds": ccds, "points": points, "prior": prior, "one": one, "seed": seed}


# ---------------------------------------------------------------- a pass
def _as(mode, x):
    return np.asarray(x, np.float32 if mode == "fp32" else np.float64)


def run(state):
    case, model, ccds = state["case"], state["model"], state["ccds"]
    mode = case["mode"]
    if case["components"] > 1:
        mix = w.MixtureModel([model(p) for p in state["points"]], state["prior"])
        total, grads, dprior = mix.gradient(ccds, mode=mode)
        return [{"total": _as(mode, total), "gradient": _as(mode, np.stack(grads)), "prior": _as(mode, dprior)}]
    out = []
    for p in state["points"]:
        wm = model(p)
        if case["op"] == "logl":
            got = w.logpdf(wm, ccds[0], mode=mode) if state["one"] else w.logpdf_families(wm, ccds, mode=mode)
            out.append({"families": _as(mode, got).reshape(-1)})
            continue
        total, grad, fam = w.gradient(wm, ccds, mode=mode)
        r = {"total": _as(mode, total), "gradient": _as(mode, grad), "families": _as(mode, fam)}
        if case["samples"]:
            trees = w.backtrack(wm, ccds, n=case["samples"], seed=state["seed"], cap=1024)
            nodes = np.full((len(trees), case["samples"], 1024, 4), -2, np.int32)  # one shape for every draw
            for i, ts in enumerate(trees):
                for j, t in enumerate(ts):
                    nodes[i, j, :len(t)] = t.nodes
            r["nodes"] = nodes
        out.append(r)
    return out


# ---------------------------------------------------------------- the tree, and what a pass needs
class _Node:
    def __init__(self):
        self.kids, self.name, self.length, self.id, self.bits = [], "", math.nan, 0, 0


def _parse(newick):
    """Newick to nodes in postorder, numbered as the models number them:
    leaves first, then the other nodes in postorder; WGD nodes (unary) after
    all others, in preorder among themselves."""
    pos = 0

    def read():
        nonlocal pos
        d = _Node()
        if newick[pos] == "(":
            pos += 1
            while True:
                d.kids.append(read())
                pos += 1
                if newick[pos - 1] == ")":
                    break
        a = pos
        while newick[pos] not in ":,();":
            pos += 1
        d.name = newick[a:pos]
        if newick[pos] == ":":
            a = pos = pos + 1
            while newick[pos] not in ",();":
                pos += 1
            d.length = float(newick[a:pos])
        return d

    root = read()
    pre, post = [], []

    def walk(d):
        pre.append(d)
        for c in d.kids:
            walk(c)
        post.append(d)

    walk(root)
    order = [d for d in pre if not d.kids] + [d for d in post if d.kids]
    plain = [d for d in order if len(d.kids) != 1]
    for i, d in enumerate(plain + [d for d in order if len(d.kids) == 1]):
        d.id = i
    for i, d in enumerate([d for d in pre if len(d.kids) == 1]):
        d.wgd = i
    for d in order:
        d.bits = 1 << d.id if not d.kids else sum(c.bits for c in d.kids)
    return order, len(plain)


def _slices(d, dt):
    return 0 if math.isnan(d.length) else max(5, math.ceil(d.length / dt))


def _flat(fams):
    """All families' clades and splits as flat arrays, with each clade's
    species as bits."""
    base = np.cumsum([0] + [len(c) for c in fams])
    size = np.concatenate([c.size for c in fams])
    species = np.concatenate([c.leaf_species for c in fams])
    own = np.concatenate([np.repeat(np.arange(len(c)), np.diff(c.split_off)) + b for c, b in zip(fams, base)])
    a = np.concatenate([c.g1.astype(np.int64) + b for c, b in zip(fams, base)])
    b = np.concatenate([c.g2.astype(np.int64) + o for c, o in zip(fams, base)])
    p = np.concatenate([c.p for c in fams])
    bits = np.zeros(len(size), np.uint64)
    leaf = size == 1
    bits[leaf] = np.uint64(1) << species[leaf].astype(np.uint64)
    by = size[own]
    for s in range(2, int(size.max()) + 1):
        at = by == s
        bits[own[at]] = bits[a[at]] | bits[b[at]]
    return base, size, own, a, b, p, bits


def _counts(case):
    """(clades, splits, cells, split terms) a family, over a sample."""
    newick, pool = _pool(case)
    order, _ = _parse(newick)
    sample = pool[:200]
    base, size, own, a, b, p, bits = _flat(sample)
    cells = terms = 0
    for d in order:
        R = _slices(d, case["dt"]) + 1
        inside = (bits & np.uint64(~d.bits & (2 ** 64 - 1))) == 0
        n, m = int(inside.sum()), int(inside[own].sum())
        cells += R * n
        terms += (R - 1 + max(0, len(d.kids))) * m
    k = len(sample)
    return len(size) / k, len(own) / k, cells / k, terms / k


def work(case):
    """Bytes: the families' CCDs read once an evaluation (8 bytes a clade, two
    clade numbers and a probability a split), a value a family written.
    Operations: two a cell, three a split term; a gradient three times that."""
    clades, splits, cells, terms = _counts(case)
    evals = case["families"] * max(case["points"], case["components"])
    grad = case["op"] == "gradient"
    return {"bytes": evals * (8 * clades + 16 * splits + 8), "flops": evals * (2 * cells + 3 * terms) * (3 if grad else 1)}


# ---------------------------------------------------------------- the same in 64 bits
def _geom(eta, x):
    return eta * x / (1 - (1 - eta) * x)


def _likelihood(order, dt, fams, flat, par, condition):
    """Per-family log-likelihoods and the conditioning term, in float64 torch
    (reference: src/core.jl:83-199, src/model.jl:162-191, src/bdputil.jl:6-11,
    src/condition.jl:11-29), all families of a node at once."""
    lam, mu, q, eta = par
    base, size, own, a, b, p, bits = flat
    size_t, p = torch.from_numpy(size), torch.from_numpy(p)
    top, eps_top, index, where = {}, {}, {}, {}
    zero = torch.zeros(1, dtype=torch.float64)

    def of(child, clades):  # top values of a child's branch, 0 where a clade does not fit it
        i = index[child.id][clades]
        return torch.cat([top[child.id], zero])[torch.from_numpy(i)]

    for d in order:
        inside = np.nonzero((bits & np.uint64(~d.bits & (2 ** 64 - 1))) == 0)[0]
        idx = np.full(len(size), len(inside), np.int64)
        idx[inside] = np.arange(len(inside))
        index[d.id] = idx
        ok = idx[own] < len(inside)
        so, sa, sb, sp = own[ok], a[ok], b[ok], p[torch.from_numpy(ok)]
        lo, la, lb = (torch.from_numpy(idx[x]) for x in (so, sa, sb))
        n = len(inside)
        acc = lambda t: torch.zeros(n, dtype=torch.float64).index_add(0, lo, t)  # noqa: E731
        if not d.kids:
            eps = torch.zeros((), dtype=torch.float64)
            v = (size_t[torch.from_numpy(inside)] == 1).double()
        elif len(d.kids) == 1:
            f = d.kids[0]
            ef, qq = eps_top[f.id], q[d.wgd]
            eps = qq * ef * ef + (1 - qq) * ef
            F = of(f, inside)
            v = qq * acc(sp * of(f, sa) * of(f, sb)) + (1 - qq + 2 * qq * ef) * F
        else:
            f, g = d.kids
            ef, eg = eps_top[f.id], eps_top[g.id]
            eps = ef * eg
            v = acc(sp * (of(f, sa) * of(g, sb) + of(g, sa) * of(f, sb))) + eg * of(f, inside) + ef * of(g, inside)
        if math.isnan(d.length):  # the root: its own smaller clades too, by size
            xi = 1 - (1 - eta) * eps
            v = v * (eta * (1 - eps) / xi ** 2)
            by = torch.from_numpy(size[so])
            for s in range(2, int(size.max()) + 1):
                at = by == s
                if bool(at.any()):
                    v = v.index_add(0, lo[at], sp[at] * v[la[at]] * v[lb[at]] * ((1 - eta) * xi / eta))
            last = torch.from_numpy(idx[base[1:] - 1])
            ll = torch.log(v[last])
            if condition == "root":
                c = torch.log(1 - _geom(eta, ef) - _geom(eta, eg) + _geom(eta, eps))
            elif condition == "nonextinct":
                c = torch.log(1 - _geom(eta, eps))
            else:
                c = torch.zeros((), dtype=torch.float64)
            return ll, c
        k = _slices(d, dt)
        t = d.length / k
        e = d
        while len(e.kids) == 1:  # a WGD node takes the rates of the branch below it
            e = e.kids[0]
        L, M = lam[e.id], mu[e.id]
        E = torch.exp(t * (L - M))
        al = M * (E - 1) / (L * E - M)
        be = L / M * al
        for _ in range(k):
            den = 1 - be * eps
            phi = (1 - al) * (1 - be) / den ** 2
            psi = phi * be / den
            eps = (al + (1 - al - be) * eps) / den
            v = phi * v + psi * acc(sp * v[la] * v[lb])
        top[d.id], eps_top[d.id] = v, eps


def exact(case, seed):
    clades, splits, cells, terms = _counts(case)
    evals = case["families"] * max(case["points"], case["components"])
    if evals * (cells + terms) * (3 if case["op"] == "gradient" else 1) > 2.5e8:
        return None
    newick, fams, points, prior = _inputs(case, seed)
    order, n_plain = _parse(newick)
    flat = _flat(fams)

    def leaf(x):
        return torch.tensor(np.asarray(x, float), dtype=torch.float64, requires_grad=case["op"] == "gradient")

    def parameters(r):
        return [leaf(r.λ), leaf(r.μ), leaf(r.q), leaf(r.η)]

    def at(par):
        return _likelihood(order, case["dt"], fams, flat, (torch.exp(par[0]), torch.exp(par[1]), par[2], par[3]),
                           case["condition"])

    def vector(grads, par):
        return np.concatenate([(torch.zeros_like(x) if g is None else g).reshape(-1).numpy() for g, x in zip(grads, par)])

    if case["components"] > 1:
        pars, pr = [parameters(r) for r in points], leaf(prior)
        cols = []
        for j, par in enumerate(pars):
            ll, c = at(par)
            cols.append(ll + torch.log(pr[j]) - c)
        total = torch.logsumexp(torch.stack(cols, 1), 1).sum()
        grads = torch.autograd.grad(total, [x for par in pars for x in par] + [pr], allow_unused=True)
        return [{"total": total.detach().numpy(), "prior": grads[-1].numpy(),
                 "gradient": np.stack([vector(grads[4 * j:4 * j + 4], pars[j]) for j in range(len(pars))])}]
    out = []
    for r in points:
        par = parameters(r)
        ll, c = at(par)
        if case["op"] == "logl":
            out.append({"families": ll.detach().numpy()})
            continue
        total = (ll - c).sum()
        grads = torch.autograd.grad(total, par, allow_unused=True)
        o = {"total": total.detach().numpy(), "gradient": vector(grads, par), "families": ll.detach().numpy()}
        if case["samples"]:
            o.update(nodes=None)
        out.append(o)
    return out
