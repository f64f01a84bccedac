"""Input populations whose steps run several at a time.

Inside a batch the updates of a population that nothing reaches and that keeps no
state run up to 16 steps per launch; a run of one step uses the ordinary update.
Both have to give the same values, spikes and records, whatever the lengths (20:
launches of 16 and 4; 9: one, launched step by step the first time and captured
from the second on; 33: a batch, then 13).

Which statements qualify is decided by the generator: a value read before the
step assigns it keeps its population out.
"""

import numpy as np
import pytest

import annarchy_amd as ah
from annarchy_amd import codegen
from annarchy_amd import connectivity as conn

SinRate = ah.Neuron(parameters="phase = 0.0", equations="r = 0.5 + 0.5*sin(0.1*t + phase)", name="SinRate")
SumRate = ah.Neuron(equations="r = sum(exc)", name="SumRate")
PoissonPre = ah.Neuron(parameters="rates = 40.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt",
                       spike="p < rates", name="PoissonPre")
Every5 = ah.Neuron(equations="v = v + 1.0\nmp = t\nq = g_exc", spike="v == 5.0", reset="v = 0.0", name="Every5")

RUNS = (20, 9, 9, 33, 1, 40, 33)


@pytest.mark.parametrize("equations, yes", [
    ("r = 0.5 + 0.5*sin(0.1*t)", True),
    ("a = Uniform(0.0, 1.0)\nr = 2.0 * a", True),
    ("r = 2.0 * a\na = Uniform(0.0, 1.0)", False),       # reads last step's a
    ("r += 0.1", False),
    ("tau*dr/dt + r = 1.0", False),
    ("r = if t > 5: 1.0 else: r", False),
    ("r = if t > 5: 1.0 else: 0.5", True),
    ("r = sum(exc)", False),                             # a psp target
])
def test_which_statements_run_ahead(equations, yes):
    src = codegen.generate_from_text("M", "tau = 10.0", equations, None, None, None).source
    assert ("void ahead_update" in src) == yes


def _rate(pre_size, post_size, precision):
    rng = np.random.default_rng(pre_size)
    k = min(3, pre_size)
    net = ah.Network(dt=1.0, seed=3, precision=precision)
    inp, pop = net.create(pre_size, SinRate), net.create(post_size, SumRate)
    for delays in (None, 4.0, rng.integers(1, 6, post_size * k).astype(float)):
        col = np.concatenate([np.sort(rng.choice(pre_size, k, replace=False)) for _ in range(post_size)])
        csr = conn.from_arrays(post_size, pre_size, np.arange(post_size + 1) * k, col, rng.normal(size=post_size * k))
        net.connect(inp, pop, "exc").from_csr(csr, storage_format="csr", **({} if delays is None else {"delays": delays}))
    mons = [net.monitor(pop, ["r"], capacity=64), net.monitor(inp, ["r", "phase"], capacity=64)]
    net.compile(graph_batch=20)
    inp.phase = np.linspace(0.0, 2.0, pre_size)
    return net, inp, pop, mons


@pytest.mark.gpu
@pytest.mark.parametrize("pre_size, post_size", [(1, 3), (64, 5), (257, 300)])
@pytest.mark.parametrize("precision", ["double", "float"])
def test_rates_ahead_are_the_steps(gpu, pre_size, post_size, precision):
    many, one = _rate(pre_size, post_size, precision), _rate(pre_size, post_size, precision)
    for steps in RUNS:
        many[0].run(steps)
        for _ in range(steps):
            one[0].run(1)
        for a, b in zip(many[3], one[3]):
            np.testing.assert_array_equal(a.get("r"), b.get("r"))
        np.testing.assert_array_equal(many[1].r, one[1].r)
    np.testing.assert_array_equal(many[2].r, one[2].r)


def _spiking(n, uniform_delay):
    net = ah.Network(dt=1.0, seed=5)
    inp, pop = net.create(n, PoissonPre), net.create(300, Every5)
    proj = net.connect(inp, pop, "exc")
    rng = np.random.default_rng(n)
    k = min(4, n)
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for _ in range(300)])
    csr = conn.from_arrays(300, n, np.arange(301) * k, col, np.full(300 * k, 0.5))
    proj.from_csr(csr, **({"delays": uniform_delay} if uniform_delay else {}))
    mons = [net.monitor(inp, ["spike", "p"], capacity=64), net.monitor(pop, ["q"], capacity=64),
            net.monitor(inp, ["spike"], capacity=64)]
    net.compile(graph_batch=20)
    inp.rates = np.linspace(50.0, 400.0, n)
    return net, inp, mons


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 64, 257, 4100])
@pytest.mark.parametrize("uniform_delay", [0.0, 3.0])
def test_spikes_ahead_are_the_steps(gpu, n, uniform_delay):
    many, one = _spiking(n, uniform_delay), _spiking(n, uniform_delay)
    for steps in RUNS:
        many[0].run(steps)
        for _ in range(steps):
            one[0].run(1)
        for k, name in ((0, "p"), (1, "q")):
            np.testing.assert_array_equal(many[2][k].get(name), one[2][k].get(name))
        for k in (0, 2):
            a, b = many[2][k].get("spike"), one[2][k].get("spike")
            assert a == b if isinstance(a, dict) else np.array_equal(a, b)
        np.testing.assert_array_equal(many[1].p, one[1].p)


def _deferred(n, m, capacity):
    """Spikes that a scatter reads from the mask, compacted 16 steps at a time."""
    net = ah.Network(dt=1.0, seed=5)
    pre, pop = net.create(n, Every5), net.create(m, Every5)
    rng = np.random.default_rng(n)
    k = min(3, n)
    for w in (0.5, 0.25):
        col = np.sort(rng.integers(0, n // k, (m, k)) + np.arange(k) * (n // k), axis=1).reshape(-1)
        net.connect(pre, pop, "exc").from_csr(conn.from_arrays(m, n, np.arange(m + 1) * k, col, np.full(m * k, w)))
    mons = [net.monitor(pre, ["spike"], capacity=capacity), net.monitor(pop, ["q", "spike"], capacity=capacity)]
    net.compile(graph_batch=20)
    # spikes in every block and in few of them
    pre.v = np.where(np.arange(n) % 7 < 3, np.arange(n) % 5.0, 5.0 * (np.arange(n) >= n // 2) - 40.0)
    pop.v = np.arange(m) % 5.0
    return net, pop, mons


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 64, 257, 4100, 20011, 131072, 131073])
def test_spikes_read_from_the_mask(gpu, n):
    many, one = _deferred(n, 300, sum(RUNS)), _deferred(n, 300, sum(RUNS))
    for steps in RUNS:
        many[0].run(steps)
        for _ in range(steps):
            one[0].run(1)
        np.testing.assert_array_equal(many[2][1].get("q", keep=True), one[2][1].get("q", keep=True))
        for a, b in zip(many[2], one[2]):
            for x, y in zip(a.raw_spikes(), b.raw_spikes()):
                np.testing.assert_array_equal(x, y)


@pytest.mark.gpu
def test_a_full_monitor_keeps_its_rows(gpu):
    # rows 24 on are not recorded: inside a launch of 16 steps, then all of them
    many, one = _deferred(300, 300, 24), _deferred(300, 300, 24)
    for steps in (20, 9, 20):
        many[0].run(steps)
        for _ in range(steps):
            one[0].run(1)
        for a, b in zip(many[2], one[2]):
            assert a.get("spike", keep=True) == b.get("spike", keep=True)


STDP_A = ah.STDP(tau_plus=20.0, tau_minus=20.0, A_plus=0.01, A_minus=0.0105, w_min=0.0, w_max=1.0)
# reads t_pre: its input population is compacted at every step
TIME_RULE = ah.Synapse(
    parameters="""
        tau_pre = 10.0 : projection
        tau_post = 10.0 : projection
        cApre = 0.01 : projection
        cApost = 0.0105 : projection
        wmax = 0.01 : projection
    """,
    pre_spike="""
        g_target += w
        w = clip(w - cApost * exp((t_post - t)/tau_post) , 0.0 , wmax)
    """,
    post_spike="""
        w = clip(w + cApre * exp((t_pre - t)/tau_pre) , 0.0 , wmax)
    """,
    name="TimeDependent",
)
PoissonPostG = ah.Neuron(parameters="rates = 30.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt\nmp = g_exc",
                         spike="p < rates", name="PoissonPostG")


def _plastic(synapse, n):
    net = ah.Network(dt=1.0, seed=7)
    pre, post = net.create(n, PoissonPre), net.create(300, PoissonPostG)
    rng = np.random.default_rng(n)
    k = min(5, n)
    col = np.sort(rng.integers(0, n // k, (300, k)) + np.arange(k) * (n // k), axis=1).reshape(-1)
    proj = net.connect(pre, post, "exc", synapse=synapse).from_csr(
        conn.from_arrays(300, n, np.arange(301) * k, col, rng.uniform(0.001, 0.009, 300 * k)))
    mons = [net.monitor(pre, ["spike"], capacity=sum(RUNS)), net.monitor(post, ["spike"], capacity=sum(RUNS))]
    net.compile(graph_batch=20)
    pre.rates, post.rates = 200.0, 100.0
    return net, proj, mons


@pytest.mark.gpu
@pytest.mark.parametrize("synapse", [STDP_A, TIME_RULE], ids=["stdp", "t_pre"])
@pytest.mark.parametrize("n", [3, 300, 20011])
def test_plastic_events_from_the_mask(gpu, synapse, n):
    many, one = _plastic(synapse, n), _plastic(synapse, n)
    w0 = many[1].w.copy()
    for steps in RUNS:
        many[0].run(steps)
        for _ in range(steps):
            one[0].run(1)
        np.testing.assert_array_equal(many[1].w, one[1].w)
        for a, b in zip(many[2], one[2]):
            for x, y in zip(a.raw_spikes(), b.raw_spikes()):
                np.testing.assert_array_equal(x, y)
    assert np.any(many[1].w != w0)
