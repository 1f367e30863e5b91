"""cullst at the sizes and values where its tiled kernels can go wrong: grids
around the 32 x 8 tile, single rows and columns (a plane fit without one of
its directions), boxes whose good points lie on a line, zero offsets (a zero
basis column), infinities and NaN, boxes of even and of unequal sides."""
import numpy as np
import pytest

from tests.helpers import cull_params, make_cull_grid

pytestmark = pytest.mark.gpu

# sigma and the smoothed offsets: the oracle's FP64 sums in another form, then
# rounded to float (the tolerance of the other cull parity tests)
RTOL = 2e-6


def _run_both(device, oracle32, grids, **kw):
    (gc, ga), (oc, oa) = cull_params(*grids, **kw), cull_params(*grids, **kw)
    device.cull("st_cull_run", gc)
    oracle32.cull("st_cull_run", oc)
    assert gc.nCulled == oc.nCulled
    for k in ("offR", "offA", "type"):
        assert np.array_equal(ga[k], oa[k], equal_nan=k != "type"), k
    for k in ("sigmaR", "sigmaA", "offRS", "offAS"):
        assert np.allclose(ga[k], oa[k], rtol=RTOL, atol=1e-6, equal_nan=True), k


@pytest.mark.parametrize("nA,nR", [(1, 1), (1, 70), (70, 1), (7, 31), (8, 32), (9, 33), (17, 95)])
@pytest.mark.parametrize("box", [(3, 3), (9, 9), (4, 11)])
def test_sizes_around_the_tile(device, oracle32, nA, nR, box):
    g = make_cull_grid(max(nA, 2), max(nR, 8), seed=nA * 100 + nR, hole_frac=0.1)
    g = tuple(np.ascontiguousarray(x[:nA, :nR]) for x in g)
    _run_both(device, oracle32, g, bR=box[0], bA=box[1], nGood=2, islandThresh=3)


@pytest.mark.parametrize("kind", ["row", "column", "diagonal", "zero", "constant", "special"])
def test_degenerate_fits_and_special_values(device, oracle32, kind):
    n = 40
    rng = np.random.default_rng(5)
    r = (2.0 + 0.02 * rng.standard_normal((n, n))).astype(np.float32)
    a = (-1.0 + 0.02 * rng.standard_normal((n, n))).astype(np.float32)
    good = np.ones((n, n), bool)
    if kind == "row":
        good[:] = False
        good[20] = True
    elif kind == "column":
        good[:] = False
        good[:, 11] = True
    elif kind == "diagonal":
        good[:] = np.eye(n, dtype=bool)
    elif kind == "zero":
        r[:], a[:] = 0, 0
    elif kind == "constant":
        r[:], a[:] = 3.25, -0.5
    else:
        r[5, 5], r[6, 9], a[20, 20], a[30, 31], r[33, 3] = np.inf, np.nan, np.inf, np.nan, -np.inf
    r[~good] = a[~good] = -2e9
    with np.errstate(all="ignore"):
        _run_both(device, oracle32, (r, a, np.ones_like(r), np.ones((n, n), np.uint8)), nGood=3, bR=9, bA=9)
