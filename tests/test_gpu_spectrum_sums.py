"""Bin sums of the run-time transform's last pass (compensated pairs per wave)
against an extended-precision transform and sum of the read-back field, for
wide log bins and for linear bins, at sides that take different numbers of rows
per work-group.

Tolerance: of white noise, every mode's power is about the mean, and its
amplitude is off by at most about four roundings per binary stage of the
transform, 4 log2(L) 2^-53, its power by twice that; the 64-lane scan adds six
roundings, the pairs and the final division two more."""
import numpy as np
import pytest
import scipy.fft

import axs

pytestmark = pytest.mark.gpu


def _reference(f, nd, N, edges2):
    """mode counts and |F|^2 sums of the bins [edges2[b], edges2[b+1]) of |k|^2"""
    F = scipy.fft.rfftn(f.reshape((N,) * nd).astype(np.longdouble))
    p = F.real ** 2 + F.imag ** 2
    del F
    k = np.fft.fftfreq(N, 1 / N).round().astype(np.int64)
    kz = np.arange(N // 2 + 1)
    w = np.where((kz == 0) | (kz == N // 2), 1, 2)
    sums = np.zeros(len(edges2) - 1, np.longdouble)
    count = np.zeros(len(edges2) - 1, np.int64)
    for i in range(N if nd == 3 else 1):
        plane = p[i] if nd == 3 else p
        k2 = (k[i] ** 2 if nd == 3 else 0) + k[:, None] ** 2 + kz[None, :] ** 2
        b = np.searchsorted(edges2, k2, side="right") - 1
        ok = (b >= 0) & (b < len(sums))
        ww = np.broadcast_to(w, k2.shape)[ok]
        count += np.bincount(b[ok], ww, len(sums)).astype(np.int64)
        order = np.argsort(b[ok], kind="stable")
        v, bb = (plane[ok] * ww)[order], b[ok][order]
        start = np.flatnonzero(np.r_[True, bb[1:] != bb[:-1]]) if len(bb) else []
        if len(bb):
            sums[bb[start]] += np.add.reduceat(v, start)
    return sums, count


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nd,N", [(2, 48), (2, 250), (2, 1200), (2, 1280), (3, 16), (3, 48),
                                  (3, 64), (3, 100), (3, 150), (3, 200)])
def test_bin_sums(nd, N, precision):
    rng = np.random.default_rng(N)
    a = rng.standard_normal((2, N ** nd))
    z = np.zeros(N ** nd)
    lat = axs.Lattice(nd, N, precision=precision)
    lat.set_state(a[0], a[1], z, z, tau=1.0)
    f = lat.get_state(fields=("phi2",))["phi2"]
    tol = 2 * (4 * nd * np.log2(N) + 8) * 2.0 ** -53
    half = N // 2
    # four log bins: squared edges (N/2)^(2 b / 4), |k|^2 whole numbers
    e2 = np.ceil(np.array([float(half) ** (2 * b / 4) for b in range(4)] + [half * half]))
    sums, count = _reference(f, nd, N, np.maximum(e2, 1).astype(np.int64))
    ks, pk, cnt = lat.powerspec(binning="log", nbins=4)
    np.testing.assert_array_equal(cnt, count)
    on = count > 0
    ref = sums[on] / count[on]
    assert np.abs(pk[on] - ref).max() <= tol * ref.max()
    # unit shells, normalised by 2 pi k or 4 pi k^2 of the bin's mean k
    e2 = np.append(np.arange(1, half, dtype=np.int64) ** 2, half * half)
    sums, count = _reference(f, nd, N, e2)
    ks, pk, cnt = lat.powerspec(binning="linear")
    np.testing.assert_array_equal(cnt[:half - 1], count)
    on = np.flatnonzero(count > 0)
    k = ks[on] / (2 * np.pi / float(np.float32(N) * np.float32(0.5)))
    area = 2 * np.pi * k if nd == 2 else 4 * np.pi * k * k
    got, want = pk[on] * area / count[on], sums[on] / count[on]
    assert np.abs(got - want).max() <= (tol + 8 * 2.0 ** -53) * want.max()
    lat.close()
