"""Monitors across captured runs.

A program that simulates an interval, reads its monitors (which empties them)
and simulates the next one replays the same graphs: batches of 20 steps and, from
the second time on, the remainder of 10.  What a monitor holds then has to start
at the interval's first step, whether the population's update records it (at
most four of a population), a launch of its own, or the spike compaction.

* a rate population whose update sums its own rows, its sum and r recorded,
  r every third step as well, against the trajectory computed on the host;
* the sum in a monitor of its own, the fifth of such a population, which the
  update does not record: at every step and at every second one;
* a spike monitor that is kept while the clock is set back or forward: the rows
  from the new step on are recorded again, a full one included;
* an `Every5` population with six monitors (five values, spikes), g_exc recorded
  after the events of a one-to-one projection arrive and before the neuron's own
  step.
"""

import numpy as np
import pytest

import annarchy_amd as ah
from annarchy_amd import connectivity as conn

pytestmark = pytest.mark.gpu

SinRate = ah.Neuron(parameters="phase = 0.0", equations="r = 0.5 + 0.5*sin(0.1*t + phase)", name="SinRate")
SumRate = ah.Neuron(equations="r = sum(exc)", name="SumRate")
Every3 = ah.Neuron(equations="v = v + 1.0\nmp = t", spike="v == 3.0", reset="v = 0.0", name="Every3")
Every5 = ah.Neuron(equations="v = v + 1.0\nmp = t\nq = g_exc", spike="v == 5.0", reset="v = 0.0", name="Every5")


@pytest.mark.parametrize("n", [1, 130])
def test_rate_records_follow_the_clock(gpu, n):
    rng = np.random.default_rng(n)
    W = rng.normal(0.0, 1.0, (n, 3))
    csr = conn.from_arrays(n, 3, np.arange(n + 1) * 3, np.tile(np.arange(3), n), W.reshape(-1))
    net = ah.Network(dt=1.0, seed=1)
    inp, pop = net.create(3, SinRate), net.create(n, SumRate)
    net.connect(inp, pop, "exc").from_csr(csr, storage_format="csr")
    each = net.monitor(pop, ["r", "_sum_exc"], capacity=40)
    third = net.monitor(pop, ["r"], capacity=40, period=3.0, period_offset=1.0)
    net.compile(graph_batch=20)
    phase = np.array([0.0, 1.0, 2.0])
    inp.phase = phase
    t = 0
    for steps in (30, 30, 30, 30, 17, 20, 30):
        net.run(steps)
        x = [0.5 + 0.5 * np.sin(0.1 * (u - 1) + phase) if u > 0 else np.zeros(3) for u in range(t, t + steps)]
        r = np.array([W @ v for v in x])
        np.testing.assert_allclose(each.get("r"), r, rtol=0, atol=1e-14)
        np.testing.assert_allclose(each.get("_sum_exc"), r, rtol=0, atol=1e-14)
        rows = [u - t for u in range(t, t + steps) if u % 3 == 1]
        np.testing.assert_allclose(third.get("r"), r[rows], rtol=0, atol=1e-14)
        t += steps


@pytest.mark.parametrize("period", [1.0, 2.0])
def test_a_fifth_monitor_records_the_sum_of_its_step(gpu, period):
    n = 130
    W = np.random.default_rng(3).normal(0.0, 1.0, (n, 3))
    csr = conn.from_arrays(n, 3, np.arange(n + 1) * 3, np.tile(np.arange(3), n), W.reshape(-1))
    net = ah.Network(dt=1.0, seed=1)
    inp, pop = net.create(3, SinRate), net.create(n, SumRate)
    net.connect(inp, pop, "exc").from_csr(csr, storage_format="csr")
    r = [net.monitor(pop, ["r"], capacity=40) for _ in range(4)]
    total = net.monitor(pop, ["_sum_exc"], capacity=40, period=period)
    net.compile(graph_batch=20)
    phase = np.array([0.0, 1.0, 2.0])
    inp.phase = phase
    t = 0
    for steps in (30, 30, 30, 1):
        net.run(steps)
        x = [0.5 + 0.5 * np.sin(0.1 * (u - 1) + phase) if u > 0 else np.zeros(3) for u in range(t, t + steps)]
        s = np.array([W @ v for v in x])   # r = sum(exc)
        for m in r:
            np.testing.assert_allclose(m.get("r"), s, rtol=0, atol=1e-14)
        np.testing.assert_allclose(total.get("_sum_exc"), s[[u % int(period) == 0 for u in range(t, t + steps)]],
                                   rtol=0, atol=1e-14)
        t += steps


def test_spiking_records_follow_the_clock(gpu):
    n = 300
    net = ah.Network(dt=1.0, seed=1)
    pre, pop = net.create(n, Every3), net.create(n, Every5)
    net.connect(pre, pop, "exc").one_to_one(0.5)
    mon = net.monitor(pop, ["v", "mp", "q", "g_exc", "spike"], capacity=40)
    more = net.monitor(pop, ["v"], capacity=40)
    net.compile(graph_batch=20)
    v0, u0 = np.arange(n) % 5.0, np.arange(n) % 3.0
    pop.v, pre.v = v0, u0
    v, u, arrive, t = v0.copy(), u0.copy(), np.zeros(n, bool), 0
    for steps in (30, 30, 30, 30, 17, 30):
        net.run(steps)
        vs, gs, spikes = [], [], {r: [] for r in range(n)}
        for _ in range(steps):
            gs.append(0.5 * arrive)     # the events of step t - 1; g is 0 between steps
            v, u = v + 1.0, u + 1.0
            fired, arrive = v == 5.0, u == 3.0
            v[fired], u[arrive] = 0.0, 0.0
            for r in np.flatnonzero(fired):
                spikes[r].append(t)
            vs.append(v.copy())
            t += 1
        np.testing.assert_array_equal(mon.get("v"), np.array(vs))
        np.testing.assert_array_equal(more.get("v"), np.array(vs))
        np.testing.assert_array_equal(mon.get("g_exc"), np.array(gs))
        np.testing.assert_array_equal(mon.get("q"), np.array(gs))
        np.testing.assert_array_equal(mon.get("mp"), np.repeat(np.arange(t - steps, t)[:, None], n, 1))
        assert mon.get("spike") == spikes


@pytest.mark.parametrize("persistent", [True, False])
@pytest.mark.parametrize("capacity", [60, 400])
def test_spike_rows_are_recorded_again(gpu, persistent, capacity):
    n = 40
    net = ah.Network(dt=1.0, seed=1)
    pop = net.create(n, Every5)
    net.connect(pop, pop, "exc").one_to_one(0.5)
    mon, second = (net.monitor(pop, ["spike"], capacity=capacity) for _ in range(2))
    if persistent:
        second.pause()
    net.compile(graph_batch=20)
    assert net.uses_persistent() == persistent
    v = np.arange(n) % 7.0
    pop.v = v
    rows, t = [], 0
    for steps, to in ((45, 0), (9, 20), (37, 3), (50, 55), (20, None)):
        net.run(steps)
        for _ in range(steps):
            v = v + 1.0
            fired = v == 5.0
            v[fired] = 0.0
            rows[t:t + 1] = [np.flatnonzero(fired)]
            t += 1
        held = rows[:min(t, capacity)]
        for m in (mon,) if persistent else (mon, second):
            counts, idx = m.raw_spikes()
            np.testing.assert_array_equal(counts, [r.size for r in held])
            np.testing.assert_array_equal(idx, np.concatenate(held))
        if to is not None:
            ah._lib.check(ah._lib.lib().ahip_set_time(net._h, to))
            rows = rows[:to] + [np.zeros(0, int)] * (to - len(rows))
            t = to
