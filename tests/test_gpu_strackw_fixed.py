"""The fixed-size passes of st_corr_track_fast against its general ones: the
same stages in the same order with the same roundings, so every output and
diagnostic is equal.  Window sizes of all four transforms in both
directions, no boxcar and the two clamped ones, windows that hang over the
image, an odd number of patches (the last cross spectrum has no partner),
both sample types, and edge pads from none to a chip of four samples."""
import numpy as np
import pytest

from specklesource_amd import abi, configs, track
from tests.test_gpu_strackw import _check, _run, compare
from tests.test_oracle_strackw import stw_params

pytestmark = pytest.mark.gpu

FIELDS = ("peakI", "peakJ", "fineI", "fineJ", "cmax", "peakGap", "fineGap")


@pytest.mark.parametrize("wr,wa,edge_r,edge_a,navg_r,navg_a", [
    (128, 128, 8, 8, 2, 2),
    (192, 192, 30, 11, 1, 1),
    (256, 256, 20, 40, 0, 2),
    (384, 384, 123, 0, 2, 3),
    (128, 384, 58, 20, 5, 1),
    (384, 192, 0, 90, 2, 0),
    (256, 128, 10, 58, 1, 24),
])
@pytest.mark.parametrize("stype", [abi.ST_SAMPLE_C64, abi.ST_SAMPLE_CI16])
def test_equals_general_passes(device, monkeypatch, wr, wa, edge_r, edge_a, navg_r, navg_a, stype):
    n = 560
    s = configs._spec(n, n, 7 + wr + wa, dr0=1.7, drR=2e-3, da0=-2.4, daA=3e-3, gmin=0.7, gmax=0.9, gLr=n / 1.2,
                      gLa=n / 1.4)
    par = stw_params(128, n, n, 8, navg=2, step=160, rShiftPoly=[1.7, 2e-3, 0], aShiftPoly=[-2.4, 0, 3e-3],
                     wR=wr, wA=wa, wRa=wr, wAa=wa, edgePadR=edge_r, edgePadA=edge_a, navgR=navg_r, navgA=navg_a,
                     rStart=wr // 2 + 9, aStart=wa // 2 + 9, deltaR=170, deltaA=180, nR=3, nA=3)
    a, b = track.synth_host(s)
    if stype == abi.ST_SAMPLE_CI16:
        a, b = (np.stack([np.round(x.real * 500), np.round(x.imag * 500)], -1).astype(np.int16) for x in (a, b))
    pid = device.upload_pair(a, b, stype)
    try:
        fixed = device.corr_track_fast(pid, par, diag=True)
        monkeypatch.setenv("SPECKLE_AMD_PATH", "staged")
        general = device.corr_track_fast(pid, par, diag=True)
    finally:
        device.release_pair(pid)
    ran = int((fixed.diag["peakI"][0] > -2000).sum())
    assert ran % 2 == 1, ran
    np.testing.assert_array_equal(fixed.diag["azShift"], general.diag["azShift"])
    for k in FIELDS:
        np.testing.assert_array_equal(fixed.diag[k][0], general.diag[k][0], err_msg=k)
    for k in ("offR", "offA", "corr", "type"):
        np.testing.assert_array_equal(getattr(fixed, k), getattr(general, k), err_msg=k)
    assert (fixed.nAmp, fixed.nFail) == (general.nAmp, general.nFail)


@pytest.mark.parametrize("wr,edge", [(64, 4), (160, 20), (448, 200), (640, 30), (768, 60), (1024, 500)])
def test_coarse_correlation_widths(device, oracle32, oracle64, wr, edge):
    """The column splits of the coarse correlation outside the fixed sizes
    (1 to 8 columns a thread, 4 to 1 rows a round, a last thread with fewer
    columns) against the oracle, by the rules of test_gpu_strackw."""
    na, nr = 160, wr + 120
    s = configs._spec(nr, na, 11 + wr, dr0=1.7, drR=0.5 / nr, da0=-2.4, daA=3e-3, gmin=0.7, gmax=0.9, gLr=nr / 1.2,
                      gLa=na / 1.4)
    par = stw_params(64, nr, na, 8, navg=2, rShiftPoly=[1.7, 0, 0], aShiftPoly=[-2.4, 0, 3e-3], wR=wr, wA=64, wRa=wr,
                     wAa=64, edgePadR=edge, edgePadA=8, rStart=wr // 2 + 9, aStart=45, deltaR=90, deltaA=60, nR=2, nA=2)
    a, b = track.synth_host(s)
    g = _run(device, par, a, b)
    rep, probs = compare(g, oracle32.corr_track_fast(par, a, b, diag=True),
                         oracle64.corr_track_fast(par, a, b, diag=True))
    print("\n", rep)
    assert rep["patches"] == 4
    _check(rep, probs)
