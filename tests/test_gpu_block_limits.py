"""Where the small-lattice kernels (csrc/axs_block3d.hip) hand over to the
one-step kernels: a launch of more than 2^32 work-items cannot be made, so an
ensemble that would need one takes the one-step kernels, and the bits are
those of one-step launches."""
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
