"""The one-pass 2D string finder on components that its single-precision screen
does not trust, in both forms: zeros of both signs, subnormal, tiny and huge
values, infinities and NaN, anywhere in the lattice and at row ends, the last
site and word borders, for counts and lists of lattices and ensembles.  Flags
equal the oracle's on the read-back field."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu

# exact in single precision or rounded to a value of the same kind
VALUES = {
    "finite": [0.0, -0.0, 1e-40, -1e-40, 1e-35, -1e-35, 1e-31, 1e31, 1e35, -1e35],
    "infinite": [np.inf, -np.inf, 0.0, -0.0, 1e35, -1e-40],
    "nan": [np.nan, np.inf, -np.inf, 0.0],
}


def _field(N, seed, kind):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((2, N * N))
    vals = np.array(VALUES[kind])
    for comp in range(2):
        at = rng.integers(0, N * N, max(8, N))
        a[comp, at] = rng.choice(vals, at.size)
        # row ends, the corners, and sites around word borders
        for site in (0, N - 1, N * N - N, N * N - 1, 63, 64, 127, 511, 512):
            if site < N * N and rng.random() < 0.5:
                a[comp, site] = rng.choice(vals)
    return a[0].copy(), a[1].copy()


def _reference(lat, N, member=0):
    g = lat.get_state(member=member, fields=("phi1", "phi2"))
    return O.cores(O.axion(g["phi1"], g["phi2"]), 2, N)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", list(VALUES))
@pytest.mark.parametrize("N", [4, 8, 22, 62, 64, 66, 130, 512])
def test_flags_match_oracle(N, kind, precision):
    p1, p2 = _field(N, N, kind)
    z = np.zeros(N * N)
    lat = axs.Lattice(2, N, precision=precision)
    lat.set_state(p1, p2, z, z, tau=1.0)
    n_ref, c_ref = _reference(lat, N)
    n, c = lat.strings()
    assert n == n_ref
    np.testing.assert_array_equal(c, c_ref)
    lat.set_state(p1, p2, z, z, tau=1.0)
    counts, cores = lat.string_counts()
    assert counts[0] == n_ref
    assert cores[0] == O.num_cores2(c_ref)
    lat.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ensemble_counts(precision):
    Ns = [4, 30, 64, 128, 66, 258]
    kinds = ["finite", "infinite", "nan"] * 2
    lat = axs.Lattice(2, members=Ns, precision=precision)
    for r, (N, kind) in enumerate(zip(Ns, kinds)):
        p1, p2 = _field(N, 7 + N, kind)
        z = np.zeros(N * N)
        lat.set_state(p1, p2, z, z, member=r)
    counts, cores = lat.string_counts()
    for r, N in enumerate(Ns):
        n_ref, c_ref = _reference(lat, N, r)
        assert counts[r] == n_ref
        assert cores[r] == O.num_cores2(c_ref)
    lat.close()
