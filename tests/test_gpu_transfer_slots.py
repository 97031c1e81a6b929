"""Transfers move through 4 MiB pinned slots by a copy kernel, 16 bytes a
work-item and the last bytes one by one: round trips whose last chunk holds
one, a few or all but one of a slot's sites, and byte copies (coordinate
lists, the axion field) of every remainder of 16."""
import os
import threading

import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu


# sites of the last chunk (2^18 FP64 sites a slot): 16, 131044, 2^18, 2052; 1026^2 and
# 1182^2 span several slots
@pytest.mark.parametrize("nd,N", [(2, 4), (2, 362), (2, 512), (2, 514), (2, 1026), (2, 1182),
                                  (3, 64), (3, 66)])
def test_round_trip(nd, N):
    rng = np.random.default_rng(N)
    a = rng.standard_normal((6, N ** nd))
    lat = axs.Lattice(nd, N)
    for sign in (1.0, -1.0):
        lat.set_state(*(sign * a), tau=1.0)
        g = lat.get_state()
        for k, x in zip(lat.STATE_FIELDS, a):
            np.testing.assert_array_equal(g[k], sign * x, err_msg=k)
    g = lat.get_state(fields=("phidot1",))
    np.testing.assert_array_equal(g["phidot1"], -a[2])
    lat.close()


@pytest.mark.parametrize("N", [34, 36, 38, 40, 42, 44, 112, 114])
def test_byte_copies(N):
    # 12 bytes a coordinate row, 8 a value of the axion field
    rng = np.random.default_rng(N)
    p1, p2 = rng.standard_normal(N ** 3), rng.standard_normal(N ** 3)
    z = np.zeros(N ** 3)
    lat = axs.Lattice(3, N)
    lat.set_state(p1, p2, z, z, tau=1.0)
    ax = lat.axion()
    np.testing.assert_array_equal(ax, O.atan2_cr(p1, p2))
    n_ref, c_ref = O.cores(ax, 3, N)
    n, c = lat.strings()
    assert n == n_ref
    np.testing.assert_array_equal(c, c_ref)
    lat.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_read_backs_beside_a_snapshot(precision):
    # axs_snapshot_end unpacks on another host thread while this one reads the
    # state back: whichever comes second brings threads of its own
    N = 128
    rng = np.random.default_rng(5)
    a = rng.standard_normal((6, N ** 3))
    lat = axs.Lattice(3, N, precision=precision)
    lat.set_state(*a, tau=1.0)
    ref = lat.get_state()
    for _ in range(4):
        lat.snapshot_begin(fields=("phi1", "phi2", "phidot1", "phidot2", "ker1", "ker2"))
        got = {}
        t = threading.Thread(target=lambda: got.update(lat.snapshot_end()[0]))
        t.start()
        for _ in range(3):
            g = lat.get_state()
            for k in ref:
                np.testing.assert_array_equal(g[k], ref[k], err_msg=k)
        t.join()
        for k in ref:
            np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
    lat.close()


def test_contexts_share_their_threads():
    # each context's transfers are large enough to be shared among threads
    N = 700
    a = np.random.default_rng(6).standard_normal((4, N * N))
    lats = []
    for k in range(6):
        lat = axs.Lattice(2, N)
        lat.set_state(*a, tau=1.0)
        g = lat.get_state()
        np.testing.assert_array_equal(g["phi2"], a[1])
        lats.append(lat)
        if k == 0:
            first = len(os.listdir("/proc/self/task"))
    assert len(os.listdir("/proc/self/task")) < first + 4
    lats[0].close()                     # the others go on with the same threads
    lats[1].set_state(*-a, tau=1.0)
    np.testing.assert_array_equal(lats[1].get_state()["phi1"], -a[0])
    for lat in lats[1:]:
        lat.close()
    assert len(os.listdir("/proc/self/task")) < first
