"""3D multi-step passes over chunks of planes that do not divide the side (the
last one shorter): identical bits to one-step launches at sides around the
tile sizes and with few large divisors, for every stencil radius, both forms
and an ensemble."""
import numpy as np
import pytest

import axs

pytestmark = pytest.mark.gpu


def _state(N, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(N ** 3) for _ in range(6)]


def _run(Ns, nsteps, simple, **kw):
    lat = axs.Lattice(3, members=Ns, **kw)
    if simple:
        lat.set_kernel("simple")
    for r, N in enumerate(Ns):
        lat.set_state(*_state(N, N + r), member=r)
    lat.tau = 1.0
    lat.step(nsteps)
    return [lat.get_state(member=r) for r in range(len(Ns))]


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("N,stencil", [(64, 0), (94, 0), (106, 0), (134, 0), (82, 1), (94, 2),
                                       (74, 3)])
def test_matches_one_step(N, stencil, precision):
    nsteps = 7                       # full passes and a remainder
    a = _run([N], nsteps, False, precision=precision, stencil_setting=stencil)
    b = _run([N], nsteps, True, precision=precision, stencil_setting=stencil)
    for k in a[0]:
        np.testing.assert_array_equal(a[0][k], b[0][k], err_msg=k)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_ensemble_matches_one_step(precision):
    Ns = [64, 122, 94, 64]
    a, b = (_run(Ns, 9, s, precision=precision) for s in (False, True))
    for r in range(len(Ns)):
        for k in a[r]:
            np.testing.assert_array_equal(a[r][k], b[r][k], err_msg=f"{r} {k}")
