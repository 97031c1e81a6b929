"""Small 3D lattices (sides below 64) advance several steps per pass in cubes
of 16^3 sites (csrc/axs_block3d.hip) unless a launch shape is configured:
identical bits to one-step launches at sides below, at and beyond the cubes'
inner 8 sites, for every form, step count and ensemble (also with larger
members beside a small one), and the plain form equals the oracle."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu


def _state(N, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(N ** 3) for _ in range(6)]


def _run(Ns, nsteps, simple, **kw):
    lat = axs.Lattice(3, members=Ns, **kw)
    if simple:
        lat.set_kernel("simple")
    for r, N in enumerate(Ns):
        lat.set_state(*_state(N, 10 * N + r), member=r)
    lat.tau = 1.0
    lat.step(nsteps)
    return lat


def _assert_equal(a, b, n):
    for r in range(n):
        ga, gb = a.get_state(member=r), b.get_state(member=r)
        for k in ga:
            np.testing.assert_array_equal(ga[k], gb[k], err_msg=f"member {r} {k}")
    assert a.tau == b.tau


@pytest.mark.parametrize("form", ["fp32", "fp64", "hamiltonian"])
@pytest.mark.parametrize("N,nsteps", [(4, 5), (8, 4), (10, 9), (16, 3), (22, 1), (48, 6), (62, 6)])
def test_cubes_match_one_step(N, nsteps, form):
    kw = dict(precision="fp32" if form == "fp32" else "fp64")
    if form == "hamiltonian":
        kw["eom"] = "hamiltonian"
    _assert_equal(_run([N], nsteps, False, **kw), _run([N], nsteps, True, **kw), 1)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("Ns", [[6, 40, 22], [32] * 7, [24, 80, 64]])
def test_ensemble_cubes_match_one_step(Ns, precision):
    _assert_equal(_run(Ns, 7, False, precision=precision), _run(Ns, 7, True, precision=precision),
                  len(Ns))


@pytest.mark.parametrize("N", [24, 34])
def test_cubes_match_oracle(N):
    lat = _run([N], 10, False)
    st = O.State(*_state(N, 10 * N))
    st.run(O.params(3, N), O.Matrix(3, N), 10)
    g = lat.get_state()
    for k in ("phi1", "phi2", "phidot1", "phidot2", "ker1", "ker2"):
        np.testing.assert_array_equal(g[k], getattr(st, k), err_msg=k)
