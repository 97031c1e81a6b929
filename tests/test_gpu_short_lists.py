"""Coordinate lists of up to 256 KiB are written to pinned memory that the
context holds from its creation, longer ones to the device and copied: both
sides of that size against the oracle, between uploads and read-backs of the
same context (whose staging memory is another), and the first list of a
context made before anything else was sampled."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu

LIMIT = (256 << 10) - 256


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nd,N,short", [(2, 64, True), (2, 192, True), (2, 202, False),
                                        (3, 28, True), (3, 30, False)])
def test_lists_around_the_direct_size(nd, N, short, precision):
    rng = np.random.default_rng(N)
    a = rng.standard_normal((2, N ** nd))
    z = np.zeros(N ** nd)
    lat = axs.Lattice(nd, N, precision=precision)
    for p1, p2 in ((a[0], a[1]), (a[1], a[0])):
        lat.set_state(p1, p2, z, z, tau=1.0)
        n, c = lat.strings()
        g = lat.get_state(fields=("phi1", "phi2"))
        n_ref, c_ref = O.cores(O.axion(g["phi1"], g["phi2"]), nd, N)
        assert (n_ref * nd * 4 <= LIMIT) == short
        assert n == n_ref
        np.testing.assert_array_equal(c, c_ref)
        lat.background()                     # results through the same block
        n, c = lat.strings()
        np.testing.assert_array_equal(c, c_ref)
    lat.close()
