"""The sweep's sliced chunks with 1, 2, 4 and 8 lanes per row (chosen by the
sweep's rows and their length), at row counts that are no multiple of a slice.

Ten steps against the row kernel (mode 0: the same FP32 compensated sums, so a
step differs by a few roundings of 6e-8: 5e-6 after ten) and against the
oracle's FP64 instances (1e-4, the bar of the sweep: its input product runs on
split BF16)."""

import numpy as np
import pytest

from annarchy_amd.batched import RateSweep
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,p", [([1, 63, 65, 200], 0.05), ([129, 400, 511], 0.05), ([513, 800], 0.05),
                                     ([64, 1500], 0.12)], ids=["1lane", "2lanes", "4lanes", "8lanes"])
def test_lanes_per_row(gpu, sizes, p):
    sw = RateSweep(sizes, n_in=70, p=p, seed=len(sizes))
    steps, got = 10, {}
    for mode in (2, 0):
        b = sw.batched()
        b.set_mode(mode)
        b.run(steps, 4)
        got[mode] = b.rates()
    for i in range(sw.n_inst):
        ref = orc.sweep_instance_run(sw.recurrent[i], sw.w_in, sw.phase[:, i], sw.omega, float(sw.gains[i]), sw.tau,
                                     sw.dt, sw.r0[i], steps)
        ref = np.asarray(ref[0] if isinstance(ref, tuple) else ref).reshape(-1)
        scale = max(np.max(np.abs(ref)), 1e-3)
        assert np.max(np.abs(got[2][i] - got[0][i])) <= 5e-6 * scale
        assert np.max(np.abs(got[2][i] - ref)) <= 1e-4 * scale
