"""What the framework is measured on: simulations as a user's program runs them.

Every case is a network (or a batched sweep) that is built once and advanced by
`steps` steps per pass through the public entry points, after which the program
reads what it simulated for: rates, membrane potentials, spike trains, recorded
values or learned weights.  `prepare` builds the connectivity from the seed and
compiles the network; `run` is one pass.

Sizes come from the benchmark and the tests of this repository (COBA with 4000
neurons, in-degrees of 100 to 1000, rate networks of uneven in-degree, STDP
between Poisson populations, sweeps of rate networks with one shared input) or
lie between them.  All weights are scaled with the in-degree, so that a network
of any size works in the regime of the benchmark's.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import annarchy_amd as ah
from annarchy_amd import batched, connectivity as conn, models

DEV = "cuda"

# The neurons and synapses of the benchmark and of the known-answer tests.
SIN_RATE = ah.Neuron(parameters="phase = 0.0", equations="r = 0.5 + 0.5*sin(0.1*t + phase)", name="SinRate")
R_DEFAULT = ah.Neuron(equations="r=sum(Hebb)+sum(Oja)+sum(IBCM)", name="RDefault")
POISSON_PRE = ah.Neuron(parameters="rates = 40.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt",
                        spike="p < rates", name="PoissonPre")
POISSON_POST = ah.Neuron(parameters="rates = 30.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt\nmp = g_exc",
                         spike="p < rates", name="PoissonPostG")
PLASTIC = {"Hebb": (ah.Hebb(eta=0.0005), 1e-6), "Oja": (ah.Oja(eta=0.01, alpha=1.0), 1e-4),
           "IBCM": (ah.IBCM(eta=0.01, tau=50.0), 1e-6)}


def listed():
    return [
        # a few hundred neurons: the everyday rate model, where latency and launches count
        {"name": "rate_small", "kind": "rate", "n": 800, "degree": 80, "uneven": False, "format": "auto",
         "precision": "double", "steps": 400},
        # a mid-size rate network in single precision
        {"name": "rate_mid_f32", "kind": "rate", "n": 10007, "degree": 300, "uneven": False, "format": "auto",
         "precision": "float", "steps": 200},
        # the benchmark's rate network with lognormal in-degrees, at a fifth of its synapses: bandwidth
        {"name": "rate_large", "kind": "rate", "n": 40001, "degree": 500, "uneven": True, "format": "auto",
         "precision": "double", "steps": 50},
        # all-to-all connectivity, the default of small cortical models (kept dense)
        {"name": "rate_dense", "kind": "rate", "n": 2503, "degree": 2503, "uneven": False, "format": "dense",
         "precision": "double", "steps": 200},
        # two populations with synaptic delays (one uniform, one per synapse), r recorded at every step
        {"name": "rate_delay", "kind": "rate_delay", "n": 5001, "degree": 200, "max_delay": 20, "precision": "double",
         "steps": 100},
        # rate-coded learning, the weights read back after the simulation
        {"name": "rate_plastic", "kind": "rate_plastic", "rule": "Oja", "pre": 2003, "post": 1501, "degree": 600,
         "precision": "double", "steps": 200},
        # the COBA benchmark as its authors run it
        {"name": "coba_small", "kind": "coba", "n": 4000, "degree": 80, "weights": "single", "drive": 0,
         "delays": "none", "record": False, "precision": "double", "steps": 1000},
        # five times as many neurons: too large for one workgroup, one weight per projection, Poisson drive
        {"name": "coba_mid", "kind": "coba", "n": 20003, "degree": 400, "weights": "single", "drive": 2000,
         "delays": "none", "record": False, "precision": "double", "steps": 500},
        # the scaled benchmark: a weight per synapse, delivered in the reference's order
        {"name": "coba_large", "kind": "coba", "n": 80000, "degree": 100, "weights": "uniform", "drive": 8000,
         "delays": "none", "record": False, "precision": "double", "steps": 500},
        # a delay per synapse, v and g recorded at every step
        {"name": "coba_delay", "kind": "coba", "n": 10000, "degree": 200, "weights": "single", "drive": 1000,
         "delays": "uniform", "record": True, "precision": "double", "steps": 200},
        # STDP between Poisson populations, the weights read back after the simulation
        {"name": "stdp", "kind": "stdp", "pre": 20000, "post": 10000, "degree": 200, "precision": "double",
         "steps": 500},
        # a parameter sweep: many rate networks of uneven size with one shared input, stepped together
        {"name": "sweep", "kind": "sweep", "instances": 24, "n_min": 500, "n_max": 3000, "n_in": 1000,
         "steps": 200},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["rate", "rate", "dense", "rate_delay", "rate_plastic", "coba", "coba", "stdp", "sweep"])
    precision = rng.choice(["double", "double", "float"])
    if kind == "rate":
        n = size(500, 40000)
        return {"kind": "rate", "n": n, "degree": min(size(40, 500), n // 4), "uneven": rng.random() < 0.4,
                "format": "auto", "precision": precision, "steps": rng.randrange(40, 120)}
    if kind == "dense":
        n = size(300, 2500)
        return {"kind": "rate", "n": n, "degree": n, "uneven": False, "format": "dense", "precision": precision,
                "steps": rng.randrange(40, 200)}
    if kind == "rate_delay":
        return {"kind": "rate_delay", "n": size(500, 5000), "degree": size(20, 200),
                "max_delay": rng.randrange(3, 25), "precision": precision, "steps": rng.randrange(30, 100)}
    if kind == "rate_plastic":
        return {"kind": "rate_plastic", "rule": rng.choice(["Oja", "Hebb", "IBCM"]), "pre": size(300, 2000),
                "post": size(100, 1500), "degree": size(50, 250), "precision": precision,
                "steps": rng.randrange(50, 200)}
    if kind == "coba":
        n = size(2000, 60000)
        delays = rng.choice(["none", "none", "none", "uniform"]) if n <= 10000 else "none"
        return {"kind": "coba", "n": n, "degree": size(50, 130), "weights": rng.choice(["single", "uniform"]),
                "drive": 0 if delays == "none" and rng.random() < 0.3 else n // 10, "delays": delays,
                "record": n <= 10000 and rng.random() < 0.4, "precision": precision,
                "steps": rng.randrange(100, 400)}
    if kind == "stdp":
        return {"kind": "stdp", "pre": size(1000, 20000), "post": size(500, 10000), "degree": size(50, 200),
                "precision": precision, "steps": rng.randrange(100, 500)}
    return {"kind": "sweep", "instances": rng.randrange(8, 24), "n_min": 300, "n_max": size(800, 3000),
            "n_in": size(300, 1000), "steps": rng.randrange(50, 200)}


# ---------------------------------------------------------------------------
# connectivity: `degree` draws with replacement per post neuron, duplicates
# merged, sorted (a few per mille fewer synapses than drawn when sparse)
# ---------------------------------------------------------------------------
def _generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _edges(n_post, n_pre, degree, uneven, g):
    """(row_ptr int64, columns int64) on the GPU, rows ascending, columns ascending in a row."""
    if degree >= n_pre:
        rows = torch.full((n_post,), n_pre, dtype=torch.int64, device=DEV)
        cols = torch.arange(n_pre, dtype=torch.int64, device=DEV).repeat(n_post)
    else:
        if uneven:
            z = torch.randn(n_post, dtype=torch.float64, device=DEV, generator=g)
            deg = (torch.exp(z + math.log(degree) - 0.5)).round().clamp(1, n_pre // 2).to(torch.int64)
        else:
            deg = torch.full((n_post,), degree, dtype=torch.int64, device=DEV)
        owner = torch.repeat_interleave(torch.arange(n_post, dtype=torch.int64, device=DEV), deg)
        col = torch.randint(0, n_pre, (owner.numel(),), dtype=torch.int64, device=DEV, generator=g)
        key = torch.unique(owner * n_pre + col)
        rows, cols = torch.bincount(key // n_pre, minlength=n_post), key % n_pre
    ptr = torch.zeros(n_post + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(rows, 0)
    return ptr, cols


def _normal(n, sigma, g):
    return sigma * torch.randn(n, dtype=torch.float64, device=DEV, generator=g)


def _csr(n_post, n_pre, ptr, cols, w):
    return conn.from_arrays(n_post, n_pre, ptr.cpu().numpy(), cols.to(torch.int32).cpu().numpy(), w.cpu().numpy())


def _rate_inputs(case, seed):
    n, k = case["n"], case["degree"]
    g = _generator(seed, 1)
    ptr, cols = _edges(n, n, k, case["uneven"], g)
    w = _normal(cols.numel(), 0.9 / math.sqrt(k), g)
    r0 = torch.rand(n, dtype=torch.float64, device=DEV, generator=g)
    return ptr, cols, w, r0


def _delay_inputs(case, seed):
    n, k, d = case["n"], case["degree"], case["max_delay"]
    m = max(1, n // 2)
    g = _generator(seed, 2)
    ff = _edges(n, m, max(1, k // 4), False, g)
    w_ff = _normal(ff[1].numel(), 2.0 / math.sqrt(k), g)
    rec = _edges(n, n, k, False, g)
    w_rec = _normal(rec[1].numel(), 0.9 / math.sqrt(k), g)
    delay = torch.randint(1, d + 1, (rec[1].numel(),), dtype=torch.int64, device=DEV, generator=g)
    phase = 2 * math.pi * torch.rand(m, dtype=torch.float64, device=DEV, generator=g)
    return m, ff, w_ff, rec, w_rec, delay, phase, max(2, d // 2)


def _plastic_inputs(case, seed):
    g = _generator(seed, 3)
    k = min(case["degree"], case["pre"] // 2)
    # exactly k distinct pre-synaptic neurons each, so that every seed has as many weights
    picked = torch.rand(case["post"], case["pre"], device=DEV, generator=g).topk(k, dim=1).indices
    cols = picked.sort(dim=1).values.reshape(-1)
    ptr = torch.arange(case["post"] + 1, dtype=torch.int64, device=DEV) * k
    w = (0.5 + torch.rand(cols.numel(), dtype=torch.float64, device=DEV, generator=g)) / k
    phase = 2 * math.pi * torch.rand(case["pre"], dtype=torch.float64, device=DEV, generator=g)
    return ptr, cols, w, phase


def _sweep(case, seed):
    sizes = np.linspace(case["n_min"], case["n_max"], case["instances"]).astype(np.int64)
    return batched.RateSweep(sizes, n_in=case["n_in"], p=0.05, seed=int(seed))


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def _ready(net, steps):
    net.set_graph(True, min(steps, 200))
    net.prepare_graph()


def prepare(case, seed):
    return {"rate": _prepare_rate, "rate_delay": _prepare_delay, "rate_plastic": _prepare_plastic,
            "coba": _prepare_coba, "stdp": _prepare_stdp, "sweep": _prepare_sweep}[case["kind"]](case, int(seed))


def _prepare_rate(case, seed):
    n = case["n"]
    ptr, cols, w, r0 = _rate_inputs(case, seed)
    net = ah.Network(dt=1.0, seed=seed, precision=case["precision"])
    pop = net.create(n, models.RateNoisy)
    net.connect(pop, pop, "exc").from_csr(_csr(n, n, ptr, cols, w), storage_format=case["format"])
    net.compile()
    pop.r = r0.cpu().numpy()
    _ready(net, case["steps"])
    return {"case": case, "net": net, "pop": pop}


def _prepare_delay(case, seed):
    n = case["n"]
    m, ff, w_ff, rec, w_rec, delay, phase, uniform = _delay_inputs(case, seed)
    net = ah.Network(dt=1.0, seed=seed, precision=case["precision"])
    inp = net.create(m, SIN_RATE)
    pop = net.create(n, models.RateNoisy)
    net.connect(inp, pop, "exc").from_csr(_csr(n, m, *ff, w_ff), delays=float(uniform))
    net.connect(pop, pop, "exc").from_csr(_csr(n, n, *rec, w_rec), delays=delay.cpu().numpy().astype(np.float64))
    mon = net.monitor(pop, ["r"], capacity=case["steps"])
    net.compile()
    inp.phase = phase.cpu().numpy()
    _ready(net, case["steps"])
    return {"case": case, "net": net, "pop": pop, "mon": mon}


def _prepare_plastic(case, seed):
    rule, eta = PLASTIC[case["rule"]]
    ptr, cols, w, phase = _plastic_inputs(case, seed)
    net = ah.Network(dt=1.0, seed=seed, precision=case["precision"])
    pre = net.create(case["pre"], SIN_RATE)
    post = net.create(case["post"], R_DEFAULT)
    proj = net.connect(pre, post, case["rule"], synapse=rule).from_csr(_csr(case["post"], case["pre"], ptr, cols, w))
    net.compile()
    pre.phase = phase.cpu().numpy()
    proj.eta = eta
    _ready(net, case["steps"])
    return {"case": case, "net": net, "pop": post, "proj": proj}


def _prepare_coba(case, seed):
    n, k = case["n"], case["degree"]
    ne = int(0.8 * n)
    scale = 80.0 / k   # the mean input conductance of the 4000-neuron benchmark (64 E + 16 I)
    net = ah.Network(dt=0.1, seed=seed, precision=case["precision"])
    pop = net.create(n, models.COBA)
    for view, deg, w in ((pop[:ne], int(0.8 * k), 0.6 * scale), (pop[ne:], k - int(0.8 * k), 6.7 * scale)):
        weights = w if case["weights"] == "single" else conn.Uniform(0.8 * w, 1.2 * w)
        delays = 0.0 if case["delays"] == "none" else conn.Uniform(0.5, 3.0, rng=net.rng)
        proj = net.connect(view, pop, "exc" if w < 5.0 * scale else "inh")
        if case["weights"] == "single":
            proj.fixed_probability(deg / view.size, weights, delays=delays, generator="device")
        else:
            proj.fixed_number_pre(deg, weights, delays=delays, generator="device")
    if case["drive"]:
        src = net.create(case["drive"], models.poisson_neuron(5.0))
        one = np.arange(case["drive"], dtype=np.int32)
        ptr = np.minimum(np.arange(n + 1), case["drive"]).astype(np.int64)
        net.connect(src, pop, "exc").from_csr(conn.from_arrays(n, case["drive"], ptr, one, None, 0.6))
    pop.v = conn.Uniform(-60.0, -50.0, rng=net.rng)
    spikes = net.monitor(pop, ["spike"], capacity=case["steps"])
    values = net.monitor(pop, ["v", "g_exc"], capacity=case["steps"]) if case["record"] else None
    net.compile()
    pop.I = 20.0
    _ready(net, case["steps"])
    return {"case": case, "net": net, "pop": pop, "spikes": spikes, "values": values}


def _prepare_stdp(case, seed):
    stdp = ah.STDP(tau_plus=20.0, tau_minus=20.0, A_plus=0.01, A_minus=0.0105, w_min=0.0, w_max=1.0)
    net = ah.Network(dt=1.0, seed=seed, precision=case["precision"])
    pre = net.create(case["pre"], POISSON_PRE)
    post = net.create(case["post"], POISSON_POST)
    proj = net.connect(pre, post, "exc", synapse=stdp).fixed_number_pre(case["degree"], conn.Uniform(0.2, 0.8),
                                                                        generator="device")
    net.compile()
    pre.rates = 20.0
    post.rates = 10.0
    _ready(net, case["steps"])
    return {"case": case, "net": net, "pop": post, "proj": proj}


def _prepare_sweep(case, seed):
    return {"case": case, "sweep": _sweep(case, seed).batched()}


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def _values(case, x):
    """An attribute in the precision the network holds it in (the getters widen it)."""
    return x if case.get("precision") == "double" else x.astype(np.float32)


def run(state):
    case, steps = state["case"], state["case"]["steps"]
    kind = case["kind"]
    if kind == "sweep":
        state["sweep"].run(steps)
        return {"r": [_values(case, r) for r in state["sweep"].rates()]}
    net, pop = state["net"], state["pop"]
    net.run(steps)
    if kind == "rate":
        return {"r": _values(case, pop.r), "sum": _values(case, pop.sum("exc"))}
    if kind == "rate_delay":
        return {"r": _values(case, state["mon"].get("r"))}
    if kind == "rate_plastic":
        return {"r": _values(case, pop.r), "w": _values(case, state["proj"].w)}
    if kind == "stdp":
        return {"g": _values(case, pop.g_exc), "w": _values(case, state["proj"].w)}
    counts, ranks = state["spikes"].raw_spikes()
    state["spikes"].clear()
    # the population's activity over time and every neuron's number of spikes
    out = {"per_step": counts, "per_neuron": np.bincount(ranks, minlength=pop.size), "v": _values(case, pop.v)}
    if state["values"] is not None:
        out["trace"] = {name: _values(case, state["values"].get(name)) for name in ("v", "g_exc")}
    return out


# ---------------------------------------------------------------------------
# work: what one pass cannot do without.  A step of a rate network reads every
# weight and column once (a dense projection has no columns), the rates and the
# sums; a spiking step reads and writes the neurons' state and, per delivered
# event, a rank, a weight and the conductance it changes.
# ---------------------------------------------------------------------------
def work(case):
    s = 8 if case.get("precision") == "double" else 4
    kind, steps = case["kind"], case["steps"]
    if kind == "rate":
        nnz = case["n"] * case["degree"]
        col = 0 if case["format"] == "dense" else 4
        return {"bytes": steps * (nnz * (s + col) + case["n"] * 6 * s), "flops": steps * 2.0 * nnz}
    if kind == "rate_delay":
        nnz = case["n"] * case["degree"]
        return {"bytes": steps * (nnz * (s + 4 + 2) + nnz // 4 * (s + 4) + case["n"] * 8 * s),
                "flops": steps * 2.5 * nnz}
    if kind == "rate_plastic":
        nnz = case["post"] * min(case["degree"], case["pre"] // 2)
        return {"bytes": steps * nnz * (3 * s + 4), "flops": steps * 7.0 * nnz}
    if kind == "coba":
        # about 2 spikes per neuron and second in the driven network, 20 in the small one
        rate = 20.0 if case["n"] <= 4000 else 2.0
        events = case["n"] * rate * 1e-4 * case["degree"]
        record = case["n"] * 2 * s if case["record"] else 0
        return {"bytes": steps * (case["n"] * (6 * s + 12) + events * (4 + 3 * s) + record),
                "flops": steps * 20.0 * case["n"]}
    if kind == "stdp":
        pre = case["pre"] * 0.02 * case["post"] * case["degree"] / case["pre"]
        post = case["post"] * 0.01 * case["degree"]
        return {"bytes": steps * (pre * (20 + 8 * s) + post * (24 + 6 * s)) + case["post"] * case["degree"] * 8,
                "flops": steps * 10.0 * (pre + post)}
    lo, hi, b = case["n_min"], case["n_max"], case["instances"]
    nnz = 0.05 * b * (lo * lo + lo * hi + hi * hi) / 3.0
    rows = b * (lo + hi) / 2.0
    return {"bytes": steps * (nnz * 8 + rows * 12), "flops": steps * (2.0 * nnz + 2.0 * case["n_in"] ** 2 * b)}


# ---------------------------------------------------------------------------
# exact: the same simulation in 64 bits with torch.  The spiking networks give
# none: their spike trains are whole numbers, and what one rounding changes in
# a membrane potential a later spike makes visible.
# ---------------------------------------------------------------------------
def _philox_normal(seed, stream, n, t):
    """Philox4x32-10 (Salmon et al. 2011) and the Box-Muller transform, N(0, 1) for neurons 0..n-1 of step t."""
    mask = np.uint64(0xFFFFFFFF)
    c = [np.arange(n, dtype=np.uint64), np.zeros(n, np.uint64), np.full(n, t & 0xFFFFFFFF, np.uint64),
         np.full(n, t >> 32, np.uint64)]
    k0, k1 = np.uint64(seed & 0xFFFFFFFF), np.uint64(((seed >> 32) & 0xFFFFFFFF) ^ stream)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k0, p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & mask, (k1 + np.uint64(0xBB67AE85)) & mask
    u1 = 1.0 - (((c[0] << np.uint64(32)) | c[1]) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    u2 = (((c[2] << np.uint64(32)) | c[3]) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    return torch.from_numpy(np.sqrt(-2.0 * np.log(u1)) * np.cos(2.0 * np.pi * u2)).to(DEV)


def _owner(ptr):
    return torch.repeat_interleave(torch.arange(ptr.numel() - 1, device=DEV), ptr[1:] - ptr[:-1])


def _rows_sum(n, owner, v):
    return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, owner, v)


def exact(case, seed):
    f = {"rate": _exact_rate, "rate_delay": _exact_delay, "rate_plastic": _exact_plastic,
         "sweep": _exact_sweep}.get(case["kind"])
    return None if f is None else f(case, int(seed))


def _numpy(x):
    return x.cpu().numpy()


def _exact_rate(case, seed):
    n = case["n"]
    ptr, cols, w, r = _rate_inputs(case, seed)
    owner = _owner(ptr)
    for t in range(case["steps"]):
        s = _rows_sum(n, owner, w * r[cols])
        r = (r + (-r + s + 0.1 * _philox_normal(seed, 0, n, t)) / 10.0).clamp(min=0.0)
    return {"r": _numpy(r), "sum": _numpy(s)}


def _exact_delay(case, seed):
    n, steps = case["n"], case["steps"]
    m, ff, w_ff, rec, w_rec, delay, phase, uniform = _delay_inputs(case, seed)
    own_ff, own_rec = _owner(ff[0]), _owner(rec[0])
    depth = max(case["max_delay"], uniform)
    past = torch.zeros(depth, n, dtype=torch.float64, device=DEV)   # row t mod depth: r after step t
    r = torch.zeros(n, dtype=torch.float64, device=DEV)
    out = []
    for t in range(steps):
        u = t - uniform
        x = 0.5 + 0.5 * torch.sin(0.1 * u + phase) if u >= 0 else torch.zeros_like(phase)
        s = _rows_sum(n, own_ff, w_ff * x[ff[1]])
        s = s + _rows_sum(n, own_rec, w_rec * past[(t - delay) % depth, rec[1]])
        r = (r + (-r + s + 0.1 * _philox_normal(seed, 1, n, t)) / 10.0).clamp(min=0.0)
        past[t % depth] = r
        out.append(r)
    return {"r": _numpy(torch.stack(out))}


def _exact_plastic(case, seed):
    rule, eta = case["rule"], PLASTIC[case["rule"]][1]
    ptr, cols, w, phase = _plastic_inputs(case, seed)
    owner = _owner(ptr)
    x = torch.zeros(case["pre"], dtype=torch.float64, device=DEV)
    theta = torch.zeros(case["post"], dtype=torch.float64, device=DEV)
    for t in range(case["steps"]):
        r = _rows_sum(case["post"], owner, w * x[cols])
        x = 0.5 + 0.5 * torch.sin(0.1 * t + phase)
        a, b = x[cols], r[owner]
        if rule == "Hebb":
            dw = eta * a * b
        elif rule == "Oja":
            dw = eta * (a * b - b * b * w)
        else:
            theta = theta + (1.0 - math.exp(-1.0 / 50.0)) * (r * r - theta)
            dw = eta * b * (b - theta[owner]) * a
        w = (w + dw).clamp(min=0.0)
    return {"r": _numpy(r), "w": _numpy(w)}


def _exact_sweep(case, seed):
    sw = _sweep(case, seed)
    w_in = torch.from_numpy(sw.w_in).to(DEV)
    phase = torch.from_numpy(sw.phase).to(DEV)
    off = np.concatenate([[0], np.cumsum(sw.sizes)])
    owner, cols, w, row, inst = [], [], [], [], []
    for i, c in enumerate(sw.recurrent):
        owner.append(np.repeat(np.arange(c.n_rows), np.diff(c.row_ptr)) + off[i])
        cols.append(c.col_idx.astype(np.int64) + off[i])
        w.append(c.w)
        row.append(np.arange(c.n_rows))
        inst.append(np.full(c.n_rows, i))
    owner, cols, w, row, inst = (torch.from_numpy(np.concatenate(v)).to(DEV) for v in (owner, cols, w, row, inst))
    r = torch.from_numpy(np.concatenate(sw.r0)).to(DEV)
    gain = torch.from_numpy(sw.gains).to(DEV)[inst]
    fed, row = row < sw.n_in, row.clamp(max=sw.n_in - 1)
    for t in range(case["steps"]):
        x = 1.0 + 0.5 * torch.sin(sw.omega * (t - 1) * sw.dt + phase) if t > 0 else torch.zeros_like(phase)
        y = torch.where(fed, (w_in @ x)[row, inst], 0.0)
        r = (r + sw.dt * ((_rows_sum(r.numel(), owner, w * r[cols]) + gain * y - r) / sw.tau)).clamp(min=0.0)
    return {"r": np.split(_numpy(r), off[1:-1])}
