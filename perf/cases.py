"""The work a user of this package has it do, as cases to time and compare.

Each case is a dict of plain values; its "kind" names the public entry point:

  model      Gillespie.run: the named-species API, host arrays in and out
  batch      Batch: resumable trajectories, advanced, edited on the host, advanced
  grid       GillespieNet.run_device: N trajectories sampled on a time grid
  events     GillespieNet.run_all_events_device: every event recorded (nb_steps = 0)
  system     a define_system network on the grid
  sweep      GillespieNet.run_sweep_device: rate constants and counts per point
  large      a network beyond the specialised kernels' 32 species / 64 reactions
  jobs       run_jobs: many different networks in one launch
  expr       a large network with Rate::Expr rates
  infer      the surrogate's fused inference pass
  train      the surrogate's forward pass, loss and backward pass

Simulated counts, event numbers and record times depend on the random stream,
so `exact` has no value for them; the surrogate's outputs are real functions
of their inputs, and `exact` gives those in 64 bits.
"""

from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

from rebop_amd import Gillespie, define_system, expr, networks, surrogate, workloads
from rebop_amd.engine import GillespieNet, Rate, RateExpr, run_jobs

# mean events of a trajectory per unit of time, for `work`
SIR_EVENTS = 1630.0 / 250.0
DIMER_EVENTS = 17450.0
MM_EVENTS = 5430.0 / 50.0

DIMERS = """
    k1 k2 k3 k4 k5;
    Dimers { gene, mRNA, protein, dimer }
    transcription : gene      => gene + mRNA      @ k1
    translation   : mRNA      => mRNA + protein   @ k2
    dimerization  : 2 protein => dimer            @ k3
    decay_mRNA    : mRNA      =>                  @ k4
    decay_protein : protein   =>                  @ k5
"""


def listed():
    return [
        # one trajectory through the named-species API: what rebop's own README
        # and tests do first; all latency
        dict(name="sir-model-1", kind="model", n=1, tmax=250.0, nb=250),
        # an intervention study: advance, read, edit, advance, read
        dict(name="sir-batch-4096", kind="batch", n=4096, t1=60.0, t2=140.0),
        # the repository's SIR benchmark: few trajectories, long serial chains
        dict(name="sir-grid-1e4", kind="grid", net="sir", n=10_000, tmax=250.0, nb=250, x0=False),
        # the same model with every event recorded
        dict(name="sir-events-1e4", kind="events", n=10_000, tmax=250.0),
        # the headline benchmark: gene expression with dimerisation
        dict(name="dimers-grid-1e6", kind="grid", net="dimers", n=1_000_000, tmax=1.0, nb=100, x0=False),
        # the macro DSL's network, each trajectory with its own initial counts
        dict(name="dimers-system-1e5", kind="system", n=100_000, tmax=1.0, nb=40),
        # generating the surrogate's training data (a parameter sweep)
        dict(name="mm-sweep-4096x64", kind="sweep", points=4096, per_point=64, tmax=50.0, nb=32),
        # the repository's 128-species, 512-reaction benchmark network
        dict(name="large-128x512", kind="large", species=128, reactions=512, net_seed=7, bounded=False,
             n=131_072, tmax=1.0, events=0.0, nb=20),
        # many different networks in one launch
        dict(name="jobs-256", kind="jobs", networks=256, net_seed=2026, per_net=256, lo=100.0, hi=100_000.0, nb=50),
        # a large network with Hill, exponential, min and threshold rates
        dict(name="expr-48x96", kind="expr", species=48, reactions=96, net_seed=11, n=32_768, tmax=2.0, nb=50),
        # a million distribution queries of the surrogate
        dict(name="surrogate-infer-1e6", kind="infer", queries=1_000_000, points=8192, width=512, depth=5),
        # one training batch of the surrogate
        dict(name="surrogate-train-4096", kind="train", batch=4096, points=512, width=512, depth=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """A case of the listed ones' ranges; costs are bounded by those of the
    listed cases of the same kind."""
    kind = rng.choice(["model", "batch", "grid", "grid", "events", "system", "sweep", "large", "large", "jobs",
                       "expr", "infer", "train"])
    if kind == "model":
        return dict(kind=kind, n=_log(rng, 1, 2000), tmax=rng.uniform(50.0, 250.0), nb=rng.randint(1, 250))
    if kind == "batch":
        return dict(kind=kind, n=_log(rng, 1, 20_000), t1=rng.uniform(20.0, 80.0), t2=rng.uniform(100.0, 200.0))
    if kind == "grid":
        if rng.random() < 0.5:
            return dict(kind=kind, net="sir", n=_log(rng, 1, 300_000), tmax=rng.uniform(50.0, 250.0),
                        nb=rng.randint(1, 250), x0=rng.random() < 0.5)
        return dict(kind=kind, net="dimers", n=_log(rng, 100, 700_000), tmax=rng.uniform(0.2, 1.0),
                    nb=rng.randint(1, 100), x0=rng.random() < 0.5)
    if kind == "events":
        return dict(kind=kind, n=_log(rng, 1, 40_000), tmax=rng.uniform(50.0, 250.0))
    if kind == "system":
        return dict(kind=kind, n=_log(rng, 10, 200_000), tmax=rng.uniform(0.2, 1.0), nb=rng.randint(1, 100))
    if kind == "sweep":
        return dict(kind=kind, points=_log(rng, 1, 4096), per_point=_log(rng, 1, 64), tmax=50.0,
                    nb=rng.randint(1, 32))
    if kind == "large":
        return dict(kind=kind, species=rng.randint(33, 160), reactions=rng.randint(65, 600),
                    net_seed=rng.randrange(1 << 20), bounded=True, n=_log(rng, 64, 40_000), tmax=0.0,
                    events=float(_log(rng, 50, 1000)), nb=rng.randint(1, 60))
    if kind == "jobs":
        return dict(kind=kind, networks=_log(rng, 2, 200), net_seed=rng.randrange(1 << 20),
                    per_net=_log(rng, 16, 300), lo=100.0, hi=float(_log(rng, 1000, 80_000)), nb=rng.randint(1, 60))
    if kind == "expr":
        return dict(kind=kind, species=rng.randint(33, 60), reactions=rng.randint(65, 120),
                    net_seed=rng.randrange(1 << 20), n=_log(rng, 64, 16_384), tmax=rng.uniform(0.2, 1.0),
                    nb=rng.randint(1, 60))
    if kind == "infer":
        return dict(kind=kind, queries=_log(rng, 1, 1_000_000), points=_log(rng, 1, 8192),
                    width=rng.choice([128, 256, 512]), depth=rng.randint(2, 5))
    return dict(kind=kind, batch=64 * _log(rng, 1, 64), points=_log(rng, 16, 512),
                width=rng.choice([128, 256, 512]), depth=rng.randint(2, 5))


# -- networks ---------------------------------------------------------------


@functools.lru_cache(maxsize=8)
def _large_spec(species, reactions, net_seed, bounded):
    if not bounded and (species, reactions) == (128, 512):
        return workloads.synthetic_large(net_seed)
    return networks.synthetic(species, reactions, net_seed, bounded=bounded)


@functools.lru_cache(maxsize=4)
def _job_specs(n, net_seed):
    return workloads.heterogeneous_specs(n, net_seed)


@functools.lru_cache(maxsize=8)
def _expr_spec(species, reactions, net_seed):
    spec, names, texts = workloads.expression_large(species, reactions, net_seed)
    index = {name: i for i, name in enumerate(names)}
    return spec, [None if t is None else expr.to_postfix(expr.parse(t), index, {}) for t in texts]


def _tmax_for(spec, events):
    """A time span of about `events` events at the initial propensities."""
    total = workloads.initial_total_propensity(spec)
    return events / total if total > 0 else 1.0


def _counts(nb, species, n):
    return torch.empty((nb + 1, species, n), dtype=torch.int64, device="cuda")


def _spread(x0, n, rng):
    """Initial counts of n trajectories around x0."""
    x = rng.poisson(np.asarray(x0, dtype=np.float64), size=(n, len(x0))).astype(np.int64)
    return torch.from_numpy(np.maximum(x, 1)).cuda()


# -- the surrogate's inputs ---------------------------------------------------

IN, NF, OUT, K, S, J, NB, TMAX = 64, 16, 128, 8, 4, 64, 32, 50.0


def _weights(case, seed):
    """Weights and biases as a trained network has them: He-scaled hidden
    layers, a small head whose biases hold the prior (on the CPU, float32)."""
    g = torch.Generator().manual_seed(seed)
    dims = [IN] + [case["width"]] * (case["depth"] - 1) + [OUT]
    W, b = [], []
    for l, (a, c) in enumerate(zip(dims[:-1], dims[1:])):
        w = torch.randn(a, c, generator=g) * math.sqrt(2.0 / (NF if l == 0 else a))
        v = torch.randn(c, generator=g) * 0.05
        if l == 0:
            w[NF:] = 0.0
        if l == len(dims) - 2:
            w *= 0.1
            w[:, S * 3 * K:] = 0.0
            v[S * 3 * K:] = 0.0
            for s in range(S):
                v[s * 3 * K + K: s * 3 * K + K + K // 2] += math.log(0.5)
                v[s * 3 * K + 2 * K: s * 3 * K + 3 * K] += math.log(10.0)
        W.append(w)
        b.append(v)
    return W, b


def _points(n, rng):
    rates = 10.0 ** rng.uniform(-3.0, 1.0, size=(n, 3))
    x0 = np.zeros((n, 4), dtype=np.int64)
    x0[:, 0] = rng.integers(10, 201, n)
    x0[:, 1] = rng.integers(50, 1001, n)
    return rates, x0


def _items(case, seed):
    """(rates, x0, point index, sample index) of a batch of queries, numpy."""
    rng = np.random.default_rng(seed)
    rates, x0 = _points(case["points"], rng)
    n = case["queries"] if case["kind"] == "infer" else case["batch"]
    return rates, x0, rng.integers(0, case["points"], n), rng.integers(1, NB + 1, n), rng


def _samples(case, seed):
    """Counts a Michaelis-Menten run could have: E + ES = E0, S + ES + P = S0,
    with P growing in time; [NB + 1][4][points * J] int64."""
    rates, x0, _, _, rng = _items(case, seed)
    e0, s0 = np.repeat(x0[:, 0], J), np.repeat(x0[:, 1], J)
    kc = np.repeat(rates[:, 2], J)
    out = np.zeros((NB + 1, S, len(e0)), dtype=np.int64)
    bound = rng.uniform(0.05, 0.95, size=len(e0))
    for i in range(NB + 1):
        p = rng.binomial(s0, 1.0 - np.exp(-0.05 * kc * TMAX * i / NB))
        es = rng.binomial(np.minimum(e0, s0 - p), bound)
        out[i] = np.stack([e0 - es, s0 - p - es, es, p])
    return out


def _mlp(case, seed):
    mlp = surrogate.MLP(seed=0, width=case["width"], depth=case["depth"])
    W, b = _weights(case, seed)
    for l in range(len(W)):
        mlp.W[l].copy_(W[l])
        mlp.b[l].copy_(b[l])
        mlp.Wb[l].copy_(mlp.W[l])
        surrogate.transpose_bf16(mlp.W[l], mlp.Wt[l])
        surrogate.pack_kslices(mlp.W[l], mlp.Wp[l])
    return mlp


# -- inputs -----------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case)
    rng = np.random.default_rng(seed)
    st["stream"] = torch.cuda.current_stream().cuda_stream
    if kind == "model":
        m = Gillespie()
        m.add_reaction(1e-4, ["S", "I"], ["I", "I"])
        m.add_reaction(0.01, ["I"], ["R"])
        st["model"], st["rng"] = m, int(seed)
    elif kind == "batch":
        st["net"] = networks.build(networks.sir(), seed)
        st["start"] = np.array([999, 1, 0], dtype=np.int64)
        st["infected"] = rng.integers(0, 20, case["n"])
    elif kind == "grid":
        spec = networks.sir() if case["net"] == "sir" else networks.dimers()
        st["net"] = networks.build(spec, seed)
        st["net"].prepare()
        st["x0_t"] = _spread(spec[2], case["n"], rng) if case["x0"] else None
        st["out"] = _counts(case["nb"], spec[0], case["n"])
    elif kind == "events":
        st["net"] = networks.build(networks.sir(), seed)
        st["net"].prepare()
        st["counts"] = torch.zeros(case["n"], dtype=torch.int64, device="cuda")
        # every event of this model removes a susceptible or an infected, and
        # a trajectory also records its start and its end: room for them all
        rows = case["n"] * (999 + 1000 + 2)
        st["times"] = torch.zeros(rows, dtype=torch.float64, device="cuda")
        st["states"] = torch.zeros((rows, 3), dtype=torch.int64, device="cuda")
    elif kind == "system":
        o = define_system(DIMERS).with_parameters(25.0, 1000.0, 0.001, 0.1, 1.0)
        o.seed(seed)
        o.gene = 1
        st["object"], st["net"] = o, o.network()
        st["net"].prepare()
        st["x0_t"] = _spread([1, 5, 20, 2], case["n"], rng)
        st["out"] = _counts(case["nb"], 4, case["n"])
    elif kind == "sweep":
        rates, x0 = _points(case["points"], rng)
        st["net"] = networks.build(networks.michaelis_menten(), seed)
        st["net"].prepare()
        st["rates"], st["x0_t"] = torch.from_numpy(rates).cuda(), torch.from_numpy(x0).cuda()
        st["out"] = _counts(case["nb"], 4, case["points"] * case["per_point"])
    elif kind == "large":
        spec = _large_spec(case["species"], case["reactions"], case["net_seed"], case["bounded"])
        st["net"] = networks.build(spec, seed)
        st["tmax"] = case["tmax"] or _tmax_for(spec, case["events"])
        st["out"] = _counts(case["nb"], spec[0], case["n"])
    elif kind == "jobs":
        specs = _job_specs(case["networks"], case["net_seed"])
        targets = workloads.target_events(case["networks"], case["lo"], case["hi"])
        n, nb = case["per_net"], case["nb"]
        st["out"] = torch.empty((nb + 1) * n * sum(s[0] for s in specs), dtype=torch.int64, device="cuda")
        st["jobs"], at = [], 0
        for j, (spec, net, ev) in enumerate(zip(specs, workloads.build_nets(specs, seed), targets)):
            st["jobs"].append(dict(net=net, tmax=_tmax_for(spec, ev), nb_steps=nb, n_traj=n, traj_begin=j * n,
                                   out_ptr=st["out"].data_ptr() + 8 * at, cost_hint=ev * len(spec[1])))
            at += (nb + 1) * spec[0] * n
    elif kind == "expr":
        spec, programs = _expr_spec(case["species"], case["reactions"], case["net_seed"])
        net = GillespieNet(spec[2], seed=seed)
        for pf, (k, o, d) in zip(programs, spec[1]):
            net.add_reaction(Rate.lma(k, o) if pf is None else RateExpr.from_postfix(*pf), d)
        st["net"] = net
        st["out"] = _counts(case["nb"], spec[0], case["n"])
    else:
        rates, x0, point, sample, _ = _items(case, seed)
        st["mlp"] = _mlp(case, seed)
        st["rates"], st["x0_t"] = torch.from_numpy(rates).cuda(), torch.from_numpy(x0).cuda()
        st["point"] = torch.from_numpy(point.astype(np.int32)).cuda()
        st["sample"] = torch.from_numpy(sample.astype(np.int32)).cuda()
        n = len(point)
        if kind == "infer":
            st["head"] = torch.empty((n, OUT), dtype=torch.float32, device="cuda")
        else:
            st["samples"] = torch.from_numpy(_samples(case, seed)).cuda()
            st["X"] = torch.empty((n, IN), dtype=torch.bfloat16, device="cuda")
            st["bound"] = torch.empty((n, S), dtype=torch.float32, device="cuda")
            st["grad"] = torch.zeros((n, OUT), dtype=torch.float32, device="cuda")
            st["loss"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    return st


# -- one pass ---------------------------------------------------------------


def _sampled(out, stats):
    return dict(counts=out, events=stats.events, draws=stats.draws)


def run(st):
    kind = st["kind"]
    if kind == "model":
        ds = st["model"].run({"S": 999, "I": 1}, st["tmax"], st["nb"], rng=st["rng"],
                             n_trajectories=None if st["n"] == 1 else st["n"])
        return dict(time=np.asarray(ds["time"]), **{s: np.asarray(ds[s]) for s in ("S", "I", "R")})
    if kind == "batch":
        b = st["net"].batch(st["n"])
        b.advance_until(st["t1"])
        x = b.get_species()
        moved = np.minimum(x[:, 0], st["infected"])
        x[:, 0] -= moved
        x[:, 1] += moved
        b.set_species(x)
        b.advance_until(st["t2"])
        return dict(before=x, after=b.get_species(), time=b.get_time(), draws=b.get_draws().astype(np.int64))
    if kind in ("grid", "system", "large", "expr"):
        x0 = st.get("x0_t")
        stats = st["net"].run_device(st["tmax"], st["nb"], st["n"], st["out"].data_ptr(),
                                     x0_ptr=None if x0 is None else x0.data_ptr(), stream=st["stream"])
        return _sampled(st["out"], stats)
    if kind == "events":
        net, counts = st["net"], st["counts"]
        net.run_all_events_device(st["tmax"], st["n"], counts.data_ptr(), stream=st["stream"])
        offsets = torch.cumsum(counts, 0) - counts
        net.run_all_events_device(st["tmax"], st["n"], counts.data_ptr(), offsets.data_ptr(), st["times"].data_ptr(),
                                  st["states"].data_ptr(), stream=st["stream"])
        return dict(counts=counts, times=st["times"], states=st["states"])
    if kind == "sweep":
        stats = st["net"].run_sweep_device(st["points"], st["per_point"], st["tmax"], st["nb"],
                                           st["out"].data_ptr(), rates_ptr=st["rates"].data_ptr(),
                                           x0_ptr=st["x0_t"].data_ptr(), stream=st["stream"])
        return _sampled(st["out"], stats)
    if kind == "jobs":
        return _sampled(st["out"], run_jobs(st["jobs"], stream=st["stream"]))
    mlp, stream = st["mlp"], st["stream"]
    if kind == "infer":
        surrogate.infer(mlp.Wp, mlp.b, st["point"], st["sample"], st["rates"], st["x0_t"], st["head"], stream=stream)
        return dict(head=st["head"])
    # the passes of one training step (surrogate.train), up to the gradients
    surrogate.features(st["point"], st["sample"], st["rates"], st["x0_t"], st["X"], st["bound"])
    head = mlp.forward(st["X"])
    st["grad"].zero_()
    st["loss"].zero_()
    surrogate.nb_mixture_nll(head, st["point"], st["sample"], st["samples"], st["grad"], st["loss"],
                             1.0 / (st["batch"] * J), st["bound"])
    dW, db = mlp.backward(st["grad"])
    return dict(head=head, loss=st["loss"], dhead=st["grad"], dW=dW, db=db)


# -- what a pass cannot do without --------------------------------------------


def _event_ops(reactions):
    # the sum and the search over the propensities, the logarithm, the
    # division, the two comparisons and the sums of time and choice
    return 2.0 * reactions + 6.0


def work(case):
    kind = case["kind"]
    if kind in ("model", "batch", "grid", "events", "system", "sweep"):
        n = case["points"] * case["per_point"] if kind == "sweep" else case["n"]
        t = case["t2"] if kind == "batch" else case["tmax"]
        if kind == "system" or case.get("net") == "dimers":
            species, reactions, events = 4, 5, DIMER_EVENTS * t * t
        elif kind == "sweep":
            species, reactions, events = 4, 3, MM_EVENTS * t
        else:
            species, reactions, events = 3, 2, SIR_EVENTS * t
        if kind == "batch":
            size = 8.0 * n * (4 * species + 2)
        elif kind == "events":
            size = 8.0 * n * (events * (species + 1) + 1)
        else:
            size = 8.0 * n * species * (case["nb"] + 1)
        return dict(bytes=size, flops=n * events * _event_ops(reactions))
    if kind == "large":
        events = case["events"] or 13_350.0 * case["tmax"]
        return dict(bytes=8.0 * case["n"] * case["species"] * (case["nb"] + 1),
                    flops=case["n"] * events * _event_ops(case["reactions"]))
    if kind == "jobs":
        lo, hi = case["lo"], case["hi"]
        # a tenth of the events that the initial propensities would make: the
        # networks relax from their initial counts
        events = 0.1 * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        n = case["networks"] * case["per_net"]
        return dict(bytes=8.0 * n * 33.5 * (case["nb"] + 1), flops=n * events * _event_ops(130))
    if kind == "expr":
        return dict(bytes=8.0 * case["n"] * case["species"] * (case["nb"] + 1),
                    flops=case["n"] * 640.0 * case["tmax"] * _event_ops(case["reactions"]))
    n = case["queries"] if kind == "infer" else case["batch"]
    w, d = case["width"], case["depth"]
    weights = IN * w + (d - 2) * w * w + w * OUT
    size = 8.0 * n + 56.0 * case["points"] + 4.0 * n * OUT
    if kind == "infer":
        return dict(bytes=size + 2.0 * weights, flops=2.0 * n * weights)
    return dict(bytes=size + n * (8.0 * S * J + 4.0 * OUT) + 8.0 * weights, flops=6.0 * n * weights)


# -- the surrogate in 64 bits -------------------------------------------------


def _features64(case, seed):
    rates, x0, point, sample, _ = _items(case, seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    r, x = dev(rates)[dev(point)], dev(x0)[dev(point)].double()
    t = TMAX * dev(sample).double() / NB
    lf, lb, lc = (torch.log10(r[:, i]) for i in range(3))
    e0, s0 = x[:, 0], x[:, 1]
    le, ls, lt, lk = torch.log10(e0), torch.log10(s0), torch.log10(t), torch.log10(r[:, 1] + r[:, 2])
    f = torch.stack([
        (lf + 1.0) * 0.5, (lb + 1.0) * 0.5, (lc + 1.0) * 0.5, (e0 - 105.0) / 95.0, (s0 - 525.0) / 475.0,
        2.0 * t / TMAX - 1.0, (le - 1.65) / 0.65, (ls - 2.35) / 0.65, (lt - 0.95) / 0.75, (lc + lt) / 3.0,
        (lf + le + lt - 1.6) / 3.4, (lf + ls + lt - 2.3) / 3.4, (lk - lf - ls + 2.05) / 4.65, (lb - lc) / 4.0,
        (le - ls + 0.7) / 1.3, (lc + le + lt - ls + 0.75) / 4.05], dim=1)
    X = torch.zeros((len(f), IN), dtype=torch.float64, device="cuda")
    X[:, :NF] = f
    return X, torch.stack([e0, s0, e0, s0], dim=1), point, sample


def _forward64(X, W, b):
    h = X
    for l, (w, v) in enumerate(zip(W, b)):
        h = h @ w + v
        if l < len(W) - 1:
            h = torch.relu(h)
    return h


def _nll64(head, bound, x):
    """Total negative log-likelihood of the samples x [B][S][J] under the
    mixtures: K/2 negative binomials and K/2 binomials on the bound."""
    total = head.new_zeros(())
    lg = torch.lgamma
    for s in range(S):
        h = head[:, None, s * 3 * K:(s + 1) * 3 * K]
        xs, n = x[:, s, :, None], bound[:, None, s, None]
        logit, mean, disp = h[..., :K], h[..., K:2 * K], h[..., 2 * K:]
        half = K // 2
        lmu = torch.clamp(mean[..., :half] + torch.log(n), -8.0, 9.0)
        lr = torch.clamp(disp[..., :half], -6.0, 12.0)
        r = torch.exp(lr)
        lrm = torch.log(r + torch.exp(lmu))
        nb = lg(xs + r) - lg(r) - lg(xs + 1.0) + r * (lr - lrm) + xs * (lmu - lrm)
        th = torch.clamp(mean[..., half:], -30.0, 30.0)
        neg = torch.log1p(torch.exp(-th.abs())) + torch.clamp(-th, min=0.0)
        bi = lg(n + 1.0) - lg(xs + 1.0) - lg(torch.clamp(n - xs, min=0.0) + 1.0) - xs * neg - (n - xs) * (neg + th)
        ll = torch.log_softmax(logit, dim=-1) + torch.cat([nb, bi], dim=-1)
        total = total - torch.logsumexp(ll, dim=-1).sum()
    return total


def exact(case, seed):
    if case["kind"] not in ("infer", "train"):
        return None
    W, b = _weights(case, seed)
    W, b = [w.double().cuda() for w in W], [v.double().cuda() for v in b]
    X, bound, point, sample = _features64(case, seed)
    if case["kind"] == "infer":
        heads = []
        for a in range(0, len(X), 1 << 17):
            h = _forward64(X[a:a + (1 << 17)], W, b)
            for s in range(S):
                cols = slice(s * 3 * K + K, s * 3 * K + K + K // 2)
                h[:, cols] += torch.log(bound[a:a + (1 << 17), s:s + 1])
            heads.append(h)
        return dict(head=torch.cat(heads))
    samples = torch.from_numpy(_samples(case, seed)).cuda()
    at = torch.from_numpy(point).cuda()[:, None] * J + torch.arange(J, device="cuda")
    x = samples[torch.from_numpy(sample).cuda()[:, None], :, at].permute(0, 2, 1).double()
    for p in W + b:
        p.requires_grad_(True)
    head = _forward64(X, W, b)
    head.retain_grad()
    loss = _nll64(head, bound, x)
    (loss / (case["batch"] * J)).backward()
    return dict(head=head.detach(), loss=loss.detach().reshape(1), dhead=head.grad, dW=[w.grad for w in W],
                db=[v.grad for v in b])
