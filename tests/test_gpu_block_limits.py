"""Where the small-lattice kernels (csrc/axs_block3d.hip) hand over to the
one-step kernels: a launch of more than 2^32 work-items cannot be made, so an
ensemble that would need one takes the one-step kernels, as do FP64 ensembles
whose cubes would run in too many rounds; the bits are those of one-step
launches on either side."""
import numpy as np
import pytest

import axs

pytestmark = pytest.mark.gpu


def _state(N, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(N ** 3) for _ in range(6)]


def _equal(a, b):
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


def test_more_cubes_than_a_launch_takes():
    # 2 x 128^3 + 6^3 = 4194520 cubes of 1024 work-items, against 2^22
    s = _state(48, 1)
    one = axs.Lattice(3, 48, precision="fp32")
    one.set_kernel("simple")
    one.set_state(*s, tau=1.0)
    one.step(2)
    lat = axs.Lattice(3, members=[1024, 1024, 48], precision="fp32")
    for r in range(2):
        lat.init("kinv", seed=r + 1, member=r)
    lat.set_state(*s, member=2)
    lat.tau = 1.0
    lat.step(2)
    _equal(lat.get_state(member=2), one.get_state())
    lat.close()


# one, two, three and four rounds of one cube per CU, cubes half empty
# (20^3), and one round more than the cubes run
@pytest.mark.parametrize("Ns", [[20] * 9, [20] * 37, [48], [48] * 2, [48] * 4, [30, 64],
                                [16] * 128, [40] * 9])
def test_fp64_rounds(Ns):
    out = []
    for simple in (False, True):
        lat = axs.Lattice(3, members=Ns)
        if simple:
            lat.set_kernel("simple")
        for r, N in enumerate(Ns):
            lat.set_state(*_state(N, 10 * N + r), member=r)
        lat.tau = 1.0
        lat.step(6)
        out.append([lat.get_state(member=r) for r in range(len(Ns))])
        lat.close()
    for a, b in zip(*out):
        _equal(a, b)
