"""A launch shape read with axs_get_kernel_config and written back changes
nothing: small lattices keep the several-steps-per-pass kernels that run until
another shape is set, and the shape a context was created with brings them
back.  Which kernel runs is seen from the number of launches a step call may
make (AXS_STEP_FAIL_AFTER)."""
import numpy as np
import pytest

import axs

pytestmark = pytest.mark.gpu

NAMES = {v: k for k, v in axs.KERNELS.items()}


def _lattice(nd, N, launches, monkeypatch, **kw):
    monkeypatch.setenv("AXS_STEP_FAIL_AFTER", str(launches))
    lat = axs.Lattice(nd, N, **kw)
    monkeypatch.delenv("AXS_STEP_FAIL_AFTER")
    rng = np.random.default_rng(N)
    lat.set_state(*[rng.standard_normal(N ** nd) for _ in range(4)], tau=1.0)
    return lat


# (lattice, steps, launches of the kernels for small lattices): one-step
# launches or the fourth-order strips (two steps a launch) need more
@pytest.mark.parametrize("nd,N,kw,steps,launches", [
    (2, 48, {}, 12, 2), (2, 48, {"precision": "fp32"}, 12, 2),
    (2, 128, {"stencil_setting": 1}, 8, 2), (3, 32, {}, 8, 2),
    (3, 32, {"precision": "fp32"}, 8, 2)])
def test_reported_shape_written_back(nd, N, kw, steps, launches, monkeypatch):
    lat = _lattice(nd, N, launches, monkeypatch, **kw)
    first = lat.kernel_config()
    back = dict(first, kernel=NAMES[first["kernel"]])
    lat.set_kernel(**back)
    assert lat.kernel_config() == first
    lat.step(steps)
    # another shape takes more launches than the limit allows
    lat.set_kernel("simple")
    with pytest.raises(axs.AxsError):
        lat.step(steps)
    lat.set_kernel(**back)
    assert lat.kernel_config() == first
    lat.step(steps)
    lat.close()
