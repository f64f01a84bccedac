"""Rate-coded populations whose update sums their own rows (one launch for psp
and update).

* a recurrent network in every row layout (CSR, SELL, dense) at the edges of a
  workgroup's rows, with empty rows, against the oracle's orc_rate_run, over
  runs between which the program sets the rates (the buffer of the last step's
  rates has to follow); and against the same network with an idle inactive
  population, which takes the separate psp and update launches;
* the form that stages the rates in LDS (a network wide enough for it);
* a model of 24 sums, whose own LDS leaves no room for the rates of 16000
  neurons that a model of few sums stages;
* a population with three targets: an undelayed CSR, a CSR with a delay per
  synapse and a dense projection with a uniform delay, against a numpy
  simulation, with a transmission pause and a disabled input in between.

Tolerances: a psp of K terms differs by at most K u sum|w r| between summation
orders (u = 1.1e-16, K <= 400, sum|w r| within 30 of the largest rate), the
update takes a tenth of it, and 20 steps of a contraction add up: 1e-11 in FP64.
FP32 rows are compensated, so a step is a few roundings of r (6e-8 each) however
long the row: 1e-5.
"""

import numpy as np
import pytest

import annarchy_amd as ah
from annarchy_amd import connectivity as conn
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SinRate = ah.Neuron(parameters="phase = 0.0", equations="r = 0.5 + 0.5*sin(0.1*t + phase)", name="SinRate")
Rate3 = ah.Neuron(parameters="tau = 10.0 : population", equations="""
    tau * dr/dt = -r + sum(exc) - sum(inh) + 0.5 * sum(mod) : min = 0.0
""", name="Rate3")
SumRate = ah.Neuron(equations="r = sum(exc)", name="SumRate")


def _csr(n_post, n_pre, k, seed):
    """Ragged rows of about k entries, every 7th row empty."""
    rng = np.random.default_rng(seed)
    deg = np.minimum(n_pre, rng.integers(0, 2 * k + 1, n_post))
    deg[::7] = 0
    return conn.random_in_degree(n_pre, n_post, rng, deg, conn.Normal(0.0, 0.9 / np.sqrt(k), rng=rng))


def _recurrent(csr, fmt, precision, noise, r0, separate):
    net = ah.Network(dt=1.0, seed=1, precision=precision)
    pop = net.create(csr.n_rows, ah.RateNoisy)
    net.connect(pop, pop, "exc").from_csr(csr, **fmt)
    if separate:
        net.create(1, SumRate).disable()
    net.compile(graph_batch=5)
    pop.r = r0
    pop.inject_random(0, noise)
    net.run(12)
    r1 = np.array(pop.r).reshape(-1)
    pop.r = r0[::-1].copy()          # the next step sums these rates
    net.run(8)
    return r1, np.array(pop.r).reshape(-1), np.array(pop.sum("exc")).reshape(-1)


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("fmt", [dict(storage_format="csr"), dict(storage_format="sell", lanes=1),
                                 dict(storage_format="sell", lanes=16, sigma=64), dict(storage_format="dense")],
                         ids=lambda f: "-".join(str(v) for v in f.values()))
@pytest.mark.parametrize("n,k", [(1, 1), (3, 2), (28, 9), (29, 9), (449, 5), (1003, 60), (130, 100)])
def test_recurrent_rows(gpu, n, k, fmt, precision):
    csr = _csr(n, n, k, 10 * n + k)
    rng = np.random.default_rng(n)
    noise, r0 = rng.normal(0.0, 0.1, (20, n)), rng.random(n)
    tol = 1e-11 if precision == "double" else 1e-5
    got = _recurrent(csr, fmt, precision, noise, r0, False)
    sep = _recurrent(csr, fmt, precision, noise, r0, True)
    a, _, _ = orc.rate_run(csr.row_ptr, csr.col_idx, csr.w, r0, 10.0, 1.0, noise[:12], 12)
    b, s, _ = orc.rate_run(csr.row_ptr, csr.col_idx, csr.w, r0[::-1].copy(), 10.0, 1.0, noise[12:], 8)
    for x, y, ref in zip(got, sep, (a, b, s)):
        scale = max(1.0, np.max(np.abs(ref)))
        np.testing.assert_allclose(x, ref, rtol=0, atol=tol * scale)
        np.testing.assert_allclose(x, y, rtol=0, atol=tol * scale)


@pytest.mark.parametrize("fmt", [dict(storage_format="csr"), dict(storage_format="sell", lanes=16, sigma=1024)],
                         ids=["csr", "sell"])
def test_staged_rates(gpu, fmt):
    n = 9001
    csr = _csr(n, n, 150, 5)
    rng = np.random.default_rng(2)
    noise, r0 = rng.normal(0.0, 0.1, (20, n)), rng.random(n)
    got = _recurrent(csr, fmt, "double", noise, r0, False)
    b, s, _ = orc.rate_run(csr.row_ptr, csr.col_idx, csr.w, r0[::-1].copy(), 10.0, 1.0, noise[12:], 8)
    a, _, _ = orc.rate_run(csr.row_ptr, csr.col_idx, csr.w, r0, 10.0, 1.0, noise[:12], 12)
    for x, ref in zip(got, (a, b, s)):
        np.testing.assert_allclose(x, ref, rtol=0, atol=1e-11 * max(1.0, np.max(np.abs(ref))))


Sum24 = ah.Neuron(equations="r = " + " + ".join(f"sum(t{k})" for k in range(24)), name="Sum24")


def test_many_sums_beside_wide_rates(gpu):
    m, n = 8000, 8000
    net = ah.Network(dt=1.0, seed=1)
    a, b, pop = net.create(m, SinRate), net.create(m, SinRate), net.create(n, Sum24)
    rng, ref = np.random.default_rng(4), np.zeros(n)
    phases = [rng.random(m) * 6.0 for _ in range(2)]
    for pre, target, phase in ((a, "t0", phases[0]), (b, "t23", phases[1])):
        csr = conn.random_in_degree(m, n, rng, np.full(n, 150), conn.Normal(0.0, 0.1, rng=rng))
        net.connect(pre, pop, target).from_csr(csr, storage_format="csr")
        # r of step 1 enters the sums of step 2
        ref += np.bincount(np.repeat(np.arange(n), 150), minlength=n,
                           weights=csr.w * (0.5 + 0.5 * np.sin(0.1 + phase))[csr.col_idx])
    net.compile()
    a.phase, b.phase = phases
    net.run(3)
    np.testing.assert_allclose(np.asarray(pop.r).reshape(-1), ref, rtol=0, atol=1e-12 * np.max(np.abs(ref)))


def test_three_targets_with_delays(gpu):
    m, n = 90, 301
    rng = np.random.default_rng(8)
    rec, inh = _csr(n, n, 20, 1), _csr(n, m, 15, 2)
    delays = rng.integers(1, 7, inh.nnz)
    dense = rng.normal(0.0, 0.1, (n, m))
    mod = conn.from_arrays(n, m, np.arange(n + 1) * m, np.tile(np.arange(m), n), dense.reshape(-1))
    phase, r0 = rng.random(m) * 6.0, rng.random(n)
    net = ah.Network(dt=1.0, seed=1)
    inp, pop = net.create(m, SinRate), net.create(n, Rate3)
    p_exc = net.connect(pop, pop, "exc").from_csr(rec, storage_format="csr")
    net.connect(inp, pop, "inh").from_csr(inh, delays=delays.astype(np.float64))
    net.connect(inp, pop, "mod").from_csr(mod, storage_format="dense", delays=6.0)
    net.compile(graph_batch=4)
    inp.phase = phase
    pop.r = r0
    W, V = rec.dense(), np.zeros((7, n, m))
    rows = np.repeat(np.arange(n), np.diff(inh.row_ptr))
    np.add.at(V, (delays, rows, inh.col_idx), inh.w)
    past, r, x, t = [np.zeros(m) for _ in range(6)], r0.copy(), np.zeros(m), 0   # past[d - 1]: d steps ago
    for steps, transmit, fed in ((9, True, True), (5, False, True), (6, True, False), (9, True, True)):
        p_exc.transmission = transmit
        (inp.enable if fed else inp.disable)()
        net.run(steps)
        for _ in range(steps):
            exc = W @ r if transmit else np.zeros(n)
            i = sum(V[d] @ past[d - 1] for d in range(1, 7))
            r = np.maximum(r + (-r + exc - i + 0.5 * (dense @ past[5])) / 10.0, 0.0)
            if fed:
                x = 0.5 + 0.5 * np.sin(0.1 * t + phase)
                past = [x] + past[:-1]
            t += 1
        np.testing.assert_allclose(np.asarray(pop.r).reshape(-1), r, rtol=0, atol=1e-11 * max(1.0, r.max()))
        np.testing.assert_allclose(np.asarray(pop.sum("exc")).reshape(-1), exc, rtol=0, atol=1e-10)
