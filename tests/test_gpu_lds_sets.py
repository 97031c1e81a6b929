"""Single-precision 3D passes over one lattice whose rows are a whole number of
16 KiB keep one LDS set of the levels' planes (csrc/axs_march2.hpp): the bits
are those of one-step launches.  1024^3 is the one side within the site limit;
its states are compared plane-wise and through sums over all sites."""
import numpy as np
import pytest

import axs

pytestmark = pytest.mark.gpu


def test_one_set_passes_match_one_step():
    N, out = 1024, []
    for kernel in (None, "simple"):
        lat = axs.Lattice(3, N, precision="fp32")
        if kernel:
            lat.set_kernel(kernel)
        else:
            assert lat.kernel_config()["depth"] == 4
        lat.init("kinv", seed=3)
        lat.tau = 1.0
        res = []
        for steps in (8, 9, 3):          # four-step passes, 4 + 5, and a three-step pass
            lat.step(steps)
            lat.snapshot_begin(count=4 * N * N)
            res += list(lat.snapshot_end()[0].values())
            res += [lat.background(), lat.energy(), lat.string_counts()[0],
                    lat.powerspec(binning="log", nbins=64)[1]]
        out.append(res)
        lat.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
