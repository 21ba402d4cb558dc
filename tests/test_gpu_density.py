"""GPU density resampling against scipy's RegularGridInterpolator, the
routine the reference calls (conehead/conehead.py:525-533, :561-568):
linear, fill 0 outside, axes linspace(origin, origin + n * spacing, n),
meshgrid 'xy' layout.  FP64 coordinates on both sides; the float32 results
agree to one unit in the last place."""
import numpy as np
import pytest
from scipy.interpolate import RegularGridInterpolator

from conehead_amd.conehead import dose_grid_densities
from conehead_amd.density import resample
from conehead_amd.device import DeviceArray
from conehead_amd.phantom import Phantom

pytestmark = pytest.mark.gpu


def axes(origin, spacing, size):
    return [np.linspace(origin[a], origin[a] + size[a] * spacing[a], size[a])
            for a in range(3)]


def scipy_ref(dens, so, ss, dshape, do, ds, swap):
    f = RegularGridInterpolator(axes(so, ss, dens.shape), dens,
                                method="linear", bounds_error=False,
                                fill_value=0)
    lx, ly, lz = axes(do, ds, dshape)
    if swap:
        xx, yy, zz = np.meshgrid(lx, ly, lz)          # indexing='xy'
    else:
        xx, yy, zz = np.meshgrid(lx, ly, lz, indexing="ij")
    return np.float32(f((xx, yy, zz)))


@pytest.mark.parametrize("swap", [True, False])
def test_resample_matches_scipy(swap):
    rng = np.random.default_rng(4)
    dens = rng.random((20, 24, 18)).astype(np.float32) * 2
    so, ss = np.array([-5.0, -3.0, -4.5]), np.array([0.5, 0.4, 0.55])
    dshape = (16, 16, 12) if swap else (17, 13, 12)
    do, ds = np.array([-6.0, -2.0, -4.0]), np.array([0.71, 0.63, 0.8])
    want = scipy_ref(dens, so, ss, dshape, do, ds, swap)
    got = resample(DeviceArray.from_host(dens), dens.shape, so, ss, dshape,
                   do, ds, swap_xy=swap).download()
    assert got.shape == want.shape
    assert (want == 0).any() and (want > 0).any()      # both regimes hit
    np.testing.assert_array_max_ulp(got, want, maxulp=1)


def test_same_grid_is_the_reference_transpose():
    """On the phantom's own grid every point is a node: the result is the
    xy-transposed densities, bit for bit."""
    rng = np.random.default_rng(5)
    dens = rng.random((14, 14, 9)).astype(np.float32)
    ph = Phantom(dens, [-3.0, 0.25, -2.0], [0.5, 0.5, 0.5])
    got = resample(DeviceArray.from_host(dens), dens.shape, ph.origin,
                   ph.spacing, dens.shape, ph.origin, ph.spacing).download()
    assert np.array_equal(got, dose_grid_densities(ph))


@pytest.mark.parametrize("dz", [1, 7, 16, 17, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("swap", [True, False])
def test_lane_layouts_match_scipy(dz, swap):
    """Every width of a wavefront's row of lanes, ragged in z and in rows,
    with points outside the source; one unit in the last place as above."""
    rng = np.random.default_rng(dz)
    dens = rng.random((9, 12, 11)).astype(np.float32) * 2
    so, ss = np.array([-2.0, -3.0, -2.5]), np.array([0.5, 0.4, 0.55])
    dshape = (11, 11, dz) if swap else (13, 7, dz)
    do, ds = np.array([-2.6, -3.1, -3.0]), np.array([0.5, 0.55, 7.0 / dz])
    want = scipy_ref(dens, so, ss, dshape, do, ds, swap)
    got = resample(DeviceArray.from_host(dens), dens.shape, so, ss, dshape,
                   do, ds, swap_xy=swap).download()
    assert (want == 0).any() and (dz == 1 or (want > 0).any())
    np.testing.assert_array_max_ulp(got, want, maxulp=1)


@pytest.mark.parametrize("dshape", [
    (181, 181, 2), (250, 250, 3),      # narrow rows, one and two per lane
    (64, 65, 16), (90, 91, 17),        # rows of 16 and 32 lanes: 2 and 4
    (100, 100, 70), (97, 103, 63)])    # 8 rows, a ragged and a full width
def test_rows_per_lane_match_scipy(dshape):
    """Every count of rows per lane on grids large enough for it, ragged in
    rows; one unit in the last place as above."""
    rng = np.random.default_rng(sum(dshape))
    dens = rng.random((19, 22, 21)).astype(np.float32) * 2
    so, ss = np.array([-2.0, -3.0, -2.5]), np.array([0.5, 0.4, 0.55])
    do = np.array([-2.6, -3.1, -2.4])    # z inside the source
    ds = np.array([11.0, 9.5, 9.0]) / dshape
    want = scipy_ref(dens, so, ss, dshape, do, ds, False)
    got = resample(DeviceArray.from_host(dens), dens.shape, so, ss, dshape,
                   do, ds, swap_xy=False).download()
    assert (want == 0).any() and (want > 0).any()
    np.testing.assert_array_max_ulp(got, want, maxulp=1)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_axis_of_one_node(axis):
    """A source axis of a single node serves exactly the points on it."""
    shape = [6, 5, 4]
    shape[axis] = 1
    rng = np.random.default_rng(axis)
    dens = rng.random(shape).astype(np.float32) + 1
    o, sp = np.array([-1.0, 0.5, 2.0]), np.array([0.5, 0.5, 0.5])
    got = resample(DeviceArray.from_host(dens), dens.shape, o, sp,
                   dens.shape, o, sp, swap_xy=False).download()
    assert np.array_equal(got, dens)
    off = o.copy()
    off[axis] += 0.25
    got = resample(DeviceArray.from_host(dens), dens.shape, o, sp,
                   dens.shape, off, sp, swap_xy=False).download()
    assert (got == 0).all()
