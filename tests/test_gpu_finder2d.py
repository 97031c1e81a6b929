"""The one-pass 2D string finder (FP32 screen, FP64 decision, right-hand
corners from the next lane, words of 64 sites that cross rows): flags equal to
the oracle's on the read-back field at sides around the word, wave (512 sites)
and block (2048 sites) sizes, with zeros of both signs, tiny, huge and NaN
components, and for counts and lists of ensembles."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu


def _field(N, seed, special):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((2, N * N))
    if special:
        vals = np.array([0.0, -0.0, 1e-40, -1e-40, 1e-320, 1e35, -1e35])
        for comp in range(2):
            at = rng.integers(0, N * N, max(8, N))
            a[comp, at] = rng.choice(vals, at.size)
        both = rng.integers(0, N * N, 8)
        a[:, both] = 0.0
    return a[0].copy(), a[1].copy()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("N", [4, 6, 8, 22, 46, 62, 64, 66, 90, 128, 130, 254, 512, 1026])
def test_flags_match_oracle(N, special, precision):
    p1, p2 = _field(N, N, special and precision == "fp64")
    z = np.zeros(N * N)
    lat = axs.Lattice(2, N, precision=precision)
    lat.set_state(p1, p2, z, z, tau=1.0)
    g = lat.get_state(fields=("phi1", "phi2"))
    n_ref, c_ref = O.cores(O.axion(g["phi1"], g["phi2"]), 2, N)
    counts, cores = lat.string_counts()
    assert counts[0] == n_ref
    assert cores[0] == O.num_cores2(c_ref)
    n, c = lat.strings()
    assert n == n_ref
    np.testing.assert_array_equal(c, c_ref)
    # the list again from a context that did not count before
    lat2 = axs.Lattice(2, N, precision=precision)
    lat2.set_state(p1, p2, z, z, tau=1.0)
    n, c = lat2.strings()
    np.testing.assert_array_equal(c, c_ref)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ensemble_counts_match_single_lattices(precision):
    Ns = [4, 30, 64, 128, 66, 258]
    lat = axs.Lattice(2, members=Ns, precision=precision)
    fields = [_field(N, 7 + N, False) for N in Ns]
    for r, (N, (p1, p2)) in enumerate(zip(Ns, fields)):
        z = np.zeros(N * N)
        lat.set_state(p1, p2, z, z, member=r)
    counts, cores = lat.string_counts()
    for r, N in enumerate(Ns):
        g = lat.get_state(member=r, fields=("phi1", "phi2"))
        n_ref, c_ref = O.cores(O.axion(g["phi1"], g["phi2"]), 2, N)
        assert counts[r] == n_ref
        assert cores[r] == O.num_cores2(c_ref)


def test_nan_components():
    N = 96
    p1, p2 = _field(N, 3, False)
    p1[[5, N * 7 + N - 1, N * N - 1]] = np.nan
    z = np.zeros(N * N)
    lat = axs.Lattice(2, N)
    lat.set_state(p1, p2, z, z, tau=1.0)
    n_ref, c_ref = O.cores(O.axion(p1, p2), 2, N)
    n, c = lat.strings()
    assert n == n_ref
    np.testing.assert_array_equal(c, c_ref)


@pytest.mark.parametrize("N", [20, 48])
def test_3d_short_chunks_match_oracle(N):
    # small 3D lattices march single planes
    rng = np.random.default_rng(N)
    p1, p2 = rng.standard_normal(N ** 3), rng.standard_normal(N ** 3)
    z = np.zeros(N ** 3)
    lat = axs.Lattice(3, N)
    lat.set_state(p1, p2, z, z, tau=1.0)
    n_ref, c_ref = O.cores(O.axion(p1, p2), 3, N)
    assert lat.string_counts()[0][0] == n_ref
    n, c = lat.strings()
    np.testing.assert_array_equal(c, c_ref)
