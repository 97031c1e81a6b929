"""Small 2D lattices advance several steps per pass in 32-column blocks
(csrc/axs_block2d.hip) unless a launch shape is configured: identical bits to
one-step launches at sides below, at and beyond the blocks' edges, for every
stencil radius, form, step count and ensemble, and the plain form equals the
oracle."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu


def _state(N, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(N * N) for _ in range(6)]


def _run(Ns, nsteps, configure, **kw):
    lat = axs.Lattice(2, members=Ns, **kw)
    if configure:
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


# inner blocks: 20 (radius 1 and 3) or 16 (radius 2 and 4) columns; 52 or 48
# rows with two rows per work-item (more than 512 blocks: sides from 460 on)
@pytest.mark.parametrize("stencil", [0, 1, 2, 3])
@pytest.mark.parametrize("form", ["fp32", "fp64", "hamiltonian"])
@pytest.mark.parametrize("N,nsteps", [(4, 7), (16, 1), (20, 6), (22, 13), (34, 5), (130, 9),
                                      (470, 7)])
def test_blocks_match_one_step(N, nsteps, form, stencil):
    kw = dict(precision="fp32" if form == "fp32" else "fp64", stencil_setting=stencil)
    if form == "hamiltonian":
        kw["eom"] = "hamiltonian"
    a, b = _run([N], nsteps, False, **kw), _run([N], nsteps, True, **kw)
    _assert_equal(a, b, 1)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("Ns", [[6, 64, 22], [128] * 9 + [66], [40] * 200])
def test_ensemble_blocks_match_one_step(Ns, precision):
    a = _run(Ns, 8, False, precision=precision)
    b = _run(Ns, 8, True, precision=precision)
    _assert_equal(a, b, len(Ns))


@pytest.mark.parametrize("N,stencil", [(30, 0), (52, 1), (500, 0)])
def test_blocks_match_oracle(N, stencil):
    lat = _run([N], 8, False, stencil_setting=stencil)
    st = O.State(*_state(N, 10 * N))
    st.run(O.params(2, N, stencil_setting=stencil), O.Matrix(2, N, stencil), 8)
    g = lat.get_state()
    for k in ("phi1", "phi2", "phidot1", "phidot2", "ker1", "ker2"):
        np.testing.assert_array_equal(g[k], getattr(st, k), err_msg=k)


@pytest.mark.parametrize("N", [130, 66])
def test_strip_chunks_of_ragged_sides(N):
    # strips with chunks that do not divide the side (a configured depth)
    for precision, depth in (("fp32", 8), ("fp64", 6)):
        a = axs.Lattice(2, N, precision=precision)
        a.set_kernel("march", depth=depth)
        b = axs.Lattice(2, N, precision=precision)
        b.set_kernel("simple")
        for lat in (a, b):
            lat.set_state(*_state(N, 3), tau=1.0)
            lat.step(2 * depth)
        _assert_equal(a, b, 1)


def test_autotune_keeps_the_blocks_where_they_win():
    # the tuner's answer names the shape that would run without the blocks;
    # the context goes on with them, and the results are the same
    a, b = axs.Lattice(2, 96), axs.Lattice(2, 96)
    for lat in (a, b):
        lat.set_state(*_state(96, 5), tau=1.0)
    a.autotune(trials=4)
    assert a.kernel_config()["kernel"] in (1, 2)
    a.step(13)
    b.step(13)
    _assert_equal(a, b, 1)
