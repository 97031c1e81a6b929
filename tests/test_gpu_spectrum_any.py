"""Power spectra of sides that are no power of two (and of powers below 128) on
the library's own run-time transform: against the oracle on the read-back
field, in both forms, linear and log bins, for every radix (2, 3, 4, 5, 7, 8,
16), ragged last groups and ensembles; against the rocFFT route at larger 3D
sides; and sides with a larger prime factor, which stay with rocFFT."""
import numpy as np
import pytest

import axs
import oracle as O

pytestmark = pytest.mark.gpu


def _lattice(nd, N, precision, seed):
    rng = np.random.default_rng(seed)
    a = [rng.standard_normal(N ** nd) for _ in range(4)]
    lat = axs.Lattice(nd, N, precision=precision)
    lat.set_state(*a, tau=1.0)
    return lat


def _compare(got, ref):
    ks, pk, cnt = got
    ks_r, pk_r, cnt_r = ref
    np.testing.assert_array_equal(cnt, cnt_r)
    sel = cnt_r > 0
    np.testing.assert_allclose(pk[sel], pk_r[sel], rtol=1e-9)
    np.testing.assert_allclose(ks[sel], ks_r[sel], rtol=1e-11)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nd,N", [(2, 16), (2, 18), (2, 28), (2, 64), (2, 84), (2, 98), (2, 150),
                                  (2, 250), (2, 640), (2, 1000), (2, 2100), (2, 3000), (3, 16),
                                  (3, 20), (3, 42), (3, 64), (3, 70), (3, 96), (3, 100),
                                  (2, 34), (3, 22)])
def test_matches_oracle(nd, N, precision):
    lat = _lattice(nd, N, precision, N)
    f = lat.get_state(fields=("phi2",))["phi2"]
    _compare(lat.powerspec(binning="linear"), O.powerspec(f, nd, N, 0.5))
    _compare(lat.powerspec(binning="log", nbins=20), O.powerspec_log(f, nd, N, 0.5, 20))


@pytest.mark.parametrize("N", [192, 400])
def test_matches_rocfft(N, monkeypatch):
    out = []
    for route in ("0", "1"):
        monkeypatch.setenv("AXS_PK_ROCFFT", route)
        lat = axs.Lattice(3, N, precision="fp32")
        monkeypatch.delenv("AXS_PK_ROCFFT")
        lat.init("kinv", seed=3)
        lat.step(10)
        out.append(lat.powerspec(binning="linear"))
        lat.close()
    _compare(*out)


def test_ensemble_matches_single_lattices():
    Ns = [60, 96, 60, 48]
    rng = np.random.default_rng(1)
    fields = [[rng.standard_normal(N ** 3) for _ in range(4)] for N in Ns]
    lat = axs.Lattice(3, members=Ns)
    for r, f in enumerate(fields):
        lat.set_state(*f, member=r)
    got = lat.powerspec_all(binning="linear")
    for r, (N, f) in enumerate(zip(Ns, fields)):
        one = axs.Lattice(3, N)
        one.set_state(*f, tau=1.0)
        for x, y in zip(got[r], one.powerspec(binning="linear")):
            np.testing.assert_array_equal(x, y)
