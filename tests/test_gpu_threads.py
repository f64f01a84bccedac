"""Networks of several threads.

Each thread owns a network, runs intervals shorter than a batch, reads weights and
monitors and empties them; lengths come up twice, so that the second run of each
is captured while the other threads copy, allocate and free.  One thread builds
and destroys networks, one runs whole batches.  Nothing fails, and every network
ends as the same one run by itself."""

import threading

import numpy as np
import pytest

import annarchy_amd as ah
from annarchy_amd import connectivity as conn

pytestmark = pytest.mark.gpu

PoissonPre = ah.Neuron(parameters="rates = 40.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt",
                       spike="p < rates", name="PoissonPre")
PoissonPostG = ah.Neuron(parameters="rates = 30.0", equations="p = Uniform(0.0, 1.0) * 1000.0 / dt\nmp = g_exc",
                         spike="p < rates", name="PoissonPostG")
STDP_A = ah.STDP(tau_plus=20.0, tau_minus=20.0, A_plus=0.01, A_minus=0.0105, w_min=0.0, w_max=1.0)


def _program(seed, lengths, batch=0, again=False):
    rng = np.random.default_rng(seed)
    k = 20
    col = np.concatenate([np.sort(rng.choice(200, k, replace=False)) for _ in range(100)])
    csr = conn.from_arrays(100, 200, np.arange(101) * k, col, rng.random(100 * k))

    def build():
        net = ah.Network(dt=1.0, seed=seed)
        pre, post = net.create(200, PoissonPre), net.create(100, PoissonPostG)
        proj = net.connect(pre, post, "exc", synapse=STDP_A).from_csr(csr)
        mon = net.monitor(post, ["spike"], capacity=100)
        net.compile(allow_build=False, graph_batch=batch)
        return net, proj, mon

    net, proj, mon = build()
    out = []
    for n in lengths:
        if again:
            net.destroy()
            net, proj, mon = build()
        net.run(n)
        out += [proj.w, *mon.raw_spikes()]
        mon.clear()
    net.destroy()
    return out


def test_short_runs_in_threads(gpu):
    lengths = (10, 10, 12, 12, 14, 14, 16, 16, 18, 18, 20, 20) * 3
    jobs = [(1, lengths), (2, lengths), (3, lengths, 0, True), (4, lengths, 8)]
    alone = [_program(*job) for job in jobs]
    got, errors = {}, []

    def work(k):
        try:
            got[k] = _program(*jobs[k])
        except Exception as e:   # reported by the test's thread
            errors.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for k, ref in enumerate(alone):
        for x, y in zip(got[k], ref):
            np.testing.assert_array_equal(x, y)
