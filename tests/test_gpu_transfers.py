"""Uploads and read-backs pass through a ring of pinned slots filled and
emptied by host threads: round trips at sides around one slot, the one-thread
limit, and more chunks than slots, with arrays left out."""
import numpy as np
import pytest

import axs

pytestmark = pytest.mark.gpu


def _arrays(L, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(L) for _ in range(6)]


# 16-byte sites: 16, 131044 and 132496 (three arrays below 8 MiB: one thread),
# 2^18 (an array is one 4 MiB slot), 287496 (two, ragged) and 2985984 (three
# arrays of twelve chunks in six slots)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nd,N", [(2, 4), (2, 362), (2, 364), (2, 512), (3, 66), (3, 144)])
def test_round_trip(nd, N, precision):
    L = N ** nd
    a = _arrays(L, N)
    lat = axs.Lattice(nd, N, precision=precision)
    lat.set_state(*a, tau=1.0)
    g = lat.get_state()
    names = ("phi1", "phi2", "phidot1", "phidot2", "ker1", "ker2")
    for k, x in zip(names, a):
        if precision == "fp64":
            np.testing.assert_array_equal(g[k], x, err_msg=k)
        elif k.startswith(("phi1", "phi2", "ker")):
            np.testing.assert_array_equal(g[k], x.astype(np.float32), err_msg=k)
        else:       # u = phidot + dt/2 ker rounded once, and phidot rebuilt: 3 roundings
            assert np.abs(g[k] - x).max() < 3 * 2.0 ** -24 * 8
    # without ker (zero), and some of the arrays only
    lat.set_state(*a[:4], tau=1.0)
    g = lat.get_state(fields=("phi2", "ker1"))
    assert set(g) == {"phi2", "ker1"}
    assert not g["ker1"].any()
    ref = a[1] if precision == "fp64" else a[1].astype(np.float32)
    np.testing.assert_array_equal(g["phi2"], ref)


def test_large_list_copy():
    # a coordinate list of more than one slot (random phases: about a third
    # of the plaquettes wind)
    N = 128
    a = _arrays(N ** 3, 1)
    lat = axs.Lattice(3, N)
    lat.set_state(*a, tau=1.0)
    n, c = lat.strings()
    assert n * 12 > (4 << 20)
    flat = (c[:, 0].astype(np.int64) * N + c[:, 1]) * N + c[:, 2]
    assert np.all(np.diff(flat) > 0)
    assert n == lat.string_counts()[0][0]


def test_contexts_share_nothing():
    # two contexts in two host threads at once
    import threading
    out = {}

    def work(r):
        a = _arrays(100 ** 3, r)
        lat = axs.Lattice(3, 100)
        for _ in range(3):
            lat.set_state(*a, tau=1.0)
            g = lat.get_state()
        out[r] = all(np.array_equal(g[k], x) for k, x in zip(lat.STATE_FIELDS, a))
        lat.close()

    ts = [threading.Thread(target=work, args=(r,)) for r in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert out == {0: True, 1: True}
