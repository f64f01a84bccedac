"""Sliced tiles (sell_panel) as given and as the builder fits them to the device:
fewer tiles than half the CUs (narrower panels, rows shared by several lanes),
fewer than the CUs (lower tiles), at least as many (as asked).  One psp of ragged
rows with empty and very long ones against the dense product in float64; FP64 to
the summation bound K u sum|w r| (K <= 2000 terms: 1e-12 of the largest sum), FP32
rows are compensated: 2e-6, the bar of every psp format.

Sizes that are given are built; sizes given as upper limits, and automatic ones,
are fitted.  Weights written back, or the reported format set again, leave the
layout and so every bit of the psp as they were.
"""

import numpy as np
import pytest

import annarchy_amd as ah
from annarchy_amd import connectivity as conn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("float", 2e-6)])
@pytest.mark.parametrize("n,opts", [
    (1, dict(panel_cols=64, chunk=64)), (63, dict(panel_cols=20, chunk=64, sigma=8, lanes=2)),
    (1500, dict(panel_cols=300, chunk=2048, sigma=8, lanes=2)),     # 5 tiles
    (2000, dict(panel_cols=500, chunk=64, sigma=8, lanes=4)),       # 128
    (2900, dict(panel_cols=300, chunk=64, lanes=4)),                # 460
])
def test_tile_heights(gpu, n, opts, precision, tol):
    rng = np.random.default_rng(n)
    deg = np.minimum(n, rng.integers(0, 120, n))
    deg[::5] = 0
    deg[:: max(1, n // 7)] = min(n, 2000)
    csr = conn.random_in_degree(n, n, rng, deg, conn.Normal(0.0, 0.1, rng=rng))
    r0 = rng.random(n)
    net = ah.Network(dt=1.0, seed=3, precision=precision)
    pop = net.create(n, ah.RateNoisy)
    proj = net.connect(pop, pop, "exc").from_csr(csr, storage_format="sell_panel", **opts)
    net.compile()
    pop.r = r0
    pop.inject_random(0, np.zeros((1, n)))
    net.step()
    ref = csr.dense() @ (r0 if precision == "double" else r0.astype(np.float32).astype(np.float64))
    np.testing.assert_allclose(np.asarray(pop.sum("exc")).reshape(-1), ref, rtol=0,
                               atol=tol * max(1.0, np.max(np.abs(ref))))
    got = proj.get_format()
    panels = -(-n // opts["panel_cols"])
    assert got["panel_cols"] == -(-n // panels) and got["chunk"] == opts["chunk"]


def _one_psp(n, precision, opts, fit):
    rng = np.random.default_rng(n)
    deg = np.minimum(n, rng.integers(0, 120, n))
    deg[::5] = 0
    deg[:: max(1, n // 7)] = min(n, 2000)
    csr = conn.random_in_degree(n, n, rng, deg, conn.Normal(0.0, 0.1, rng=rng))
    r0 = rng.random(n)
    net = ah.Network(dt=1.0, seed=3, precision=precision)
    pop = net.create(n, ah.RateNoisy)
    proj = net.connect(pop, pop, "exc").from_csr(csr, storage_format="csr")
    net.compile()
    proj.set_format("sell_panel", **opts, **({"fit_tiles": True} if fit else {}))
    pop.r = r0
    pop.inject_random(0, np.zeros((1, n)))
    r = r0 if precision == "double" else r0.astype(np.float32).astype(np.float64)
    rows = np.repeat(np.arange(n), np.diff(csr.row_ptr))
    return net, pop, proj, r0, np.bincount(rows, weights=csr.w * r[csr.col_idx], minlength=n)


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("float", 2e-6)])
@pytest.mark.parametrize("n,opts,panel_cols,chunk", [
    (1500, dict(panel_cols=300, chunk=2048, sigma=8, lanes=2), 300, 64),     # 5 tiles asked: few
    (2000, dict(panel_cols=50, chunk=512, lanes=4), 50, 256),                # 160 asked: lower, not narrower
    (2900, dict(panel_cols=300, chunk=64, lanes=4), 290, 64),                # 460 asked: kept
    (15000, dict(panel_cols=15000, chunk=2048, sigma=8, lanes=2), 7500, 64), # 8 asked: narrower too
])
def test_tiles_fitted_to_the_device(gpu, n, opts, panel_cols, chunk, precision, tol):
    net, pop, proj, r0, ref = _one_psp(n, precision, opts, True)
    got = proj.get_format()
    assert (got["panel_cols"], got["chunk"]) == (panel_cols, chunk)
    net.step()
    np.testing.assert_allclose(np.asarray(pop.sum("exc")).reshape(-1), ref, rtol=0,
                               atol=tol * max(1.0, np.max(np.abs(ref))))


@pytest.mark.parametrize("opts,fit", [
    ({}, False),                                                          # automatic sizes
    (dict(panel_cols=9001, chunk=2048, sigma=8, lanes=2), False),
    (dict(panel_cols=9001, chunk=2048, sigma=8, lanes=2), True),
], ids=["automatic", "given", "limits"])
def test_a_rebuilt_layout_is_the_same(gpu, opts, fit):
    n = 9001
    net, pop, proj, r0, _ = _one_psp(n, "double", opts, fit)

    def psp():
        pop.r = r0
        net.step()
        return np.asarray(pop.sum("exc")).reshape(-1).copy()

    form, first = proj.get_format(), psp()
    assert (form["panel_cols"], form["chunk"]) == (9001, 2048 if opts and not fit else 64)
    proj.w = proj.w
    assert proj.get_format() == form
    np.testing.assert_array_equal(psp(), first)
    f = dict(form)
    proj.set_format(f.pop("format"), **f)
    assert proj.get_format() == form
    np.testing.assert_array_equal(psp(), first)
    # tiles of other sizes after them are built as given
    proj.set_format("sell_panel", panel_cols=4096, chunk=512)
    assert proj.get_format()["chunk"] == 512 and proj.get_format()["panel_cols"] == 3001
