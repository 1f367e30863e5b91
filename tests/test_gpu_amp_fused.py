"""The fused amplitude kernel against the staged kernels it stands in for.

Both run the same transforms in the same order with the same roundings, so
every try's peak, correlation and widths are equal bit for bit; the SNR
diagnostic is an FP32 sum in another order.  -noComplex runs send every point
through the small window with its own Doppler estimate, and the points that
fail it (low coherence, large shifts) through the doubled one with the shift
handed on."""
import numpy as np
import pytest

from specklesource_amd import abi, configs, track
from tests.helpers import small_params

pytestmark = pytest.mark.gpu


def _pair(na, nr, seed, stype):
    s = configs._spec(nr, na, seed, dr0=1.3, da0=-0.8, drR=3.0 / nr, gmin=0.02, gmax=0.7, gLr=nr / 2, gLa=na / 2,
                      maskR0=nr // 2, maskR1=nr // 2 + 90, maskA0=na // 3, maskA1=na // 3 + 110)
    a, b = track.synth_host(s)
    if stype == abi.ST_SAMPLE_CI16:
        a, b = (np.rint(x.view(np.float32) * 400).astype(np.int16).reshape(x.shape + (2,)) for x in (a, b))
    return a, b


@pytest.mark.parametrize("stype", [abi.ST_SAMPLE_C64, abi.ST_SAMPLE_CI16])
@pytest.mark.parametrize("w,wa", [(16, 16), (32, 32), (64, 64), (32, 16), (24, 32), (64, 128)])
def test_fused_tries_equal_staged_tries(device, monkeypatch, w, wa, stype):
    n = 20 if wa < 128 else 9
    na, nr = n * wa + 37, (n - 2) * wa + 11
    a, b = _pair(na, nr, 7 + wa, stype)
    # the grid runs over the image's edges: some small and more doubled windows are out of bounds
    p = small_params(w, nr, na, step=wa - 3, wRa=wa, wAa=wa, noComplex=1, rStart=wa // 2, aStart=wa // 2,
                     nR=(nr - wa) // (wa - 3) + 2, nA=(na - wa) // (wa - 3) + 2, rShiftPoly=[1.0, 0, 0],
                     aShiftPoly=[-1.0, 0, 0])
    pid = device.upload_pair(a, b, stype)
    try:
        f = device.speckle_track(pid, p, diag=True)
        monkeypatch.setenv("SPECKLE_AMD_PATH", "staged")
        s = device.speckle_track(pid, p, diag=True)
    finally:
        device.release_pair(pid)
    assert f.nAmp == s.nAmp > 0 and f.nAmpL == s.nAmpL and f.nFail == s.nFail > 0
    assert f.nAmpL > 0 or wa == 128
    for k in ("offR", "offA", "azd", "type"):
        assert np.array_equal(getattr(f, k), getattr(s, k)), k
    for k in ("peakI", "peakJ", "fineI", "fineJ", "sigRg", "sigAz", "peakGap", "fineGap"):
        for t in (1, 2):
            assert np.array_equal(f.diag[k][t], s.diag[k][t]), (k, t)
    # the means and powers are FP64 sums of at most 2^16 values in another order; corr rounds the same to a float ulp
    assert np.allclose(f.corr, s.corr, rtol=2**-23, atol=0)
    for t in (1, 2):
        assert np.allclose(f.diag["cmax"][t], s.diag["cmax"][t], rtol=2**16 * 2**-52, atol=0)
        # sums of at most 256^2 positive floats: 2 * 2^-24 * log2(65536) apart at most with pairwise orders, and the
        # threads' serial parts of 64 values
        assert np.allclose(f.diag["snr"][t], s.diag["snr"][t], rtol=2e-5)


@pytest.mark.parametrize("ulps", [0, 2])
@pytest.mark.parametrize("wa", [16, 32, 64])
def test_constant_windows(device, monkeypatch, wa, ulps):
    """Float windows of one value each, and such windows with a noise of units
    in the last place.  Of the former the lag sums after mean removal are zeros:
    no Doppler shift, nothing to correlate.  Of the latter they are 2^-47 of the
    windows' power, below the rounding of sums that keep the mean."""
    T, n = wa + 4, 20
    rng = np.random.default_rng(wa)

    def tiles():
        x = np.kron(rng.uniform(1, 2, (n, n, 2)).astype(np.float32), np.ones((T, T, 1), np.float32))
        k = np.float32(2**-23) * rng.integers(-ulps, ulps + 1, x.shape)
        return np.ascontiguousarray(x + k.astype(np.float32)).view(np.complex64)[..., 0]

    p = small_params(wa, n * T, n * T, step=T, wRa=wa, wAa=wa, noComplex=1, rStart=T // 2, aStart=T // 2, nR=n, nA=n,
                     maxTries=1)
    pid = device.upload_pair(tiles(), tiles())
    try:
        f = device.speckle_track(pid, p, diag=True)
        monkeypatch.setenv("SPECKLE_AMD_PATH", "staged")
        s = device.speckle_track(pid, p, diag=True)
    finally:
        device.release_pair(pid)
    assert ulps or (s.diag["peakI"][1] == -1000).all()
    for k in ("offR", "offA", "azd", "type"):
        assert np.array_equal(getattr(f, k), getattr(s, k)), k
    for k in ("peakI", "peakJ", "fineI", "fineJ", "sigRg", "sigAz", "peakGap", "fineGap"):
        assert np.array_equal(f.diag[k][1], s.diag[k][1]), k


def _both_paths(device, monkeypatch, pid, p):
    f = device.speckle_track(pid, p, diag=True)
    monkeypatch.setenv("SPECKLE_AMD_PATH", "staged")
    s = device.speckle_track(pid, p, diag=True)
    monkeypatch.delenv("SPECKLE_AMD_PATH")
    assert (f.nAmp, f.nAmpL, f.nFail) == (s.nAmp, s.nAmpL, s.nFail)
    for k in ("offR", "offA", "azd", "type"):
        assert np.array_equal(getattr(f, k), getattr(s, k)), k
    for k in ("peakI", "peakJ", "fineI", "fineJ", "sigRg", "sigAz", "peakGap", "fineGap"):
        for t in (1, 2):
            assert np.array_equal(f.diag[k][t], s.diag[k][t]), (k, t)
    assert np.allclose(f.corr, s.corr, rtol=2**-23, atol=0)  # as in test_fused_tries_equal_staged_tries
    return f


@pytest.mark.parametrize("wa,n,step", [(16, 120, 4), (32, 64, 7), (64, 32, 20)])
def test_several_tries_per_workgroup(device, monkeypatch, wa, n, step):
    """More tries than resident workgroups (at most 4096, 1024 and 256 of them),
    so that each takes three or four one after the other, with tries that leave
    early among them: windows outside the image, windows without data."""
    a, b = _pair(n * step - 9, n * step - 21, wa, abi.ST_SAMPLE_C64)
    for x in (a, b):
        x[60:150, 70:200] = 0
    p = small_params(wa, n * step, n * step, step=step, wRa=wa, wAa=wa, noComplex=1, rStart=0, aStart=0, nR=n, nA=n,
                     rShiftPoly=[1.0, 0, 0], aShiftPoly=[-1.0, 0, 0])
    pid = device.upload_pair(a, b)
    try:
        f = _both_paths(device, monkeypatch, pid, p)
    finally:
        device.release_pair(pid)
    matched = (f.diag["peakI"][1] != -2000).mean()  # tries that reached the correlation
    assert n * n > 2.5 * {16: 4096, 32: 1024, 64: 256}[wa]
    assert 0.4 < matched < 0.95 and f.nAmp > 100, matched


@pytest.mark.parametrize("w,wa", [(64, 64), (64, 128)])
def test_gauss_fits_on_the_128_sample_passes(device, monkeypatch, w, wa):
    """-gauss: the fit reads the surface that the 128 sample passes leave, of the
    doubled window or of the small one."""
    n = 14 if wa < 128 else 9
    a, b = _pair(n * wa + 37, n * wa + 11, 3 + wa, abi.ST_SAMPLE_C64)
    p = small_params(w, n * wa, n * wa, step=wa - 3, wRa=wa, wAa=wa, noComplex=1, gaussFlag=1, rStart=wa, aStart=wa,
                     nR=n - 1, nA=n - 1, rShiftPoly=[1.0, 0, 0], aShiftPoly=[-1.0, 0, 0])
    pid = device.upload_pair(a, b)
    try:
        f = _both_paths(device, monkeypatch, pid, p)
    finally:
        device.release_pair(pid)
    assert f.nAmp > 0 and (f.nAmpL > 0 or wa == 128)


def test_one_try_and_no_try(device, monkeypatch):
    """A single point, and a grid whose windows all leave the image."""
    a, b = _pair(160, 160, 3, abi.ST_SAMPLE_C64)
    pid = device.upload_pair(a, b)
    try:
        p = small_params(32, 160, 160, noComplex=1, nR=1, nA=1, rStart=50, aStart=40)
        g = _both_paths(device, monkeypatch, pid, p)
        assert g.type.shape == (1, 1) and g.diag["peakI"][1][0, 0] != -2000
        p = small_params(32, 160, 160, noComplex=1, nR=3, nA=2, rShiftPoly=[4000.0, 0, 0])
        g = device.speckle_track(pid, p)
        assert (g.type == 0).all() and g.nAmp == g.nAmpL == 0
    finally:
        device.release_pair(pid)
