"""GPU 3D-DDA traces are bit-exact with the oracle and the reference's
notebook goldens (dda_3d_c semantics, conehead/dda_3d_c.pyx:33-99)."""
import ctypes
import json
import math
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden", "dda_goldens.json")


@pytest.fixture(scope="module")
def gold():
    with open(GOLD) as f:
        return json.load(f)


def bits(a):
    return np.ascontiguousarray(a, np.float64).view(np.uint64)


def test_golden_ray_a(gold):
    from conehead_amd.dda_3d_c import dda_3d_c
    g = gold["ray_A"]
    r = math.sqrt(14.0)
    vox, t = dda_3d_c(np.array([1 / r, 2 / r, 3 / r]), g["grid_shape"],
                      g["first_voxel"], g["voxel_size"])
    expect = np.array([float(v) for v in g["t"]])
    assert np.array_equal(bits(t), bits(expect))
    assert vox[0].tolist() == [50, 50, 50]


def test_golden_ray_c(gold):
    from conehead_amd.dda_3d_c import dda_3d_c
    g = gold["ray_C"]
    d = np.array(g["direction"])
    vox, t = dda_3d_c(d, g["grid_shape"], g["first_voxel"], g["voxel_size"],
                      mutate_direction=True)
    assert vox.tolist() == g["voxels"]
    expect = np.array([[float(v) for v in s] for s in g["t_states"]]).min(1)
    assert np.array_equal(bits(t), bits(expect))
    assert d.tolist() == [0.997859, 0.0, 0.065403]   # |d| like dda_3d_c


def test_capacity_error():
    from conehead_amd import _lib
    L = _lib.lib()
    d = (ctypes.c_double * 3)(0.0, 0.0, 1.0)
    shp = (ctypes.c_int32 * 3)(4, 4, 40)
    fv = (ctypes.c_int32 * 3)(1, 1, 0)
    vs = (ctypes.c_double * 3)(1.0, 1.0, 1.0)
    vox = (ctypes.c_int32 * 30)()
    tv = (ctypes.c_double * 10)()
    n = ctypes.c_int32()
    st = L.ch_dda_3d(d, shp, fv, vs, vox, tv, 10, ctypes.byref(n), None)
    assert st == _lib.CH_ERR_CAPACITY and n.value == 40


def test_batch_matches_oracle_bitwise(oracle):
    from conehead_amd.dda_3d_c import dda_trace
    rng = np.random.default_rng(17)
    for shape, vs in [((23, 31, 17), (0.4, 0.4, 0.4)),
                      ((64, 50, 80), (0.25, 0.3, 0.2)),
                      ((7, 90, 11), (1.0, 0.1, 0.5))]:
        n = 500
        d = rng.normal(size=(n, 3))
        d[rng.random((n, 3)) < 0.1] = 0.0
        d[:5] = [[0, 0, 1], [1, 1, 1], [-1, 0, 0], [0, -0.0, 1], [1, 2, 3]]
        first = np.stack([rng.integers(0, s, size=n) for s in shape], 1)
        counts, vox, t = dda_trace(d, first, shape, vs)
        for i in range(n):
            ov, ot, _ = oracle.dda_3d(d[i], shape, first[i], vs)
            assert counts[i] == len(ot)
            assert np.array_equal(vox[i, :counts[i]], ov)
            assert np.array_equal(bits(t[i, :counts[i]]), bits(ot))


def test_terma_rays_bitwise(oracle):
    """The TERMA kernel's ray directions (voxel centre -> source, FP64) and
    traversals equal the oracle's, including oblique rays on a rotated
    gantry: FP64 alphas neither drop nor duplicate voxels."""
    from conehead_amd import _lib, engine
    from conehead_amd.device import DeviceArray
    from conehead_amd.source import Source
    from conehead_amd.workloads import SETTINGS
    shape = (96, 80, 72)
    spacing = np.array([0.25, 0.3, 0.2])
    origin = np.array([-11.9, 0.15, -7.1])
    rng = np.random.default_rng(4)
    for gantry in [0.0, 33.3, 251.0]:
        src = Source("varian_clinac_6MV")
        if gantry:
            src.gantry = gantry
        dummy = DeviceArray((16,), np.float32)
        beam = engine.beam_struct(src, SETTINGS, dummy, dummy, dummy, None)
        n = 400
        vin = np.stack([rng.integers(0, s, size=n) for s in shape], 1)
        vin = vin.astype(np.int32)
        cap = sum(shape) + 2
        d_in = DeviceArray.from_host(vin)
        d_dirs = DeviceArray((n, 3), np.float64)
        d_vox = DeviceArray((n, cap, 3), np.int32)
        d_t = DeviceArray((n, cap), np.float64)
        d_cnt = DeviceArray((n,), np.int32)
        shp = (ctypes.c_int32 * 3)(*shape)
        org = (ctypes.c_double * 3)(*origin)
        spc = (ctypes.c_double * 3)(*spacing)
        _lib.check(_lib.lib().ch_terma_rays(
            ctypes.byref(beam), shp, org, spc, n, d_in.ptr, cap, d_dirs.ptr,
            d_vox.ptr, d_t.ptr, d_cnt.ptr, None))
        dirs, vox, t, cnt = (d_dirs.download(), d_vox.download(),
                             d_t.download(), d_cnt.download())
        sp = np.asarray(src.position, np.float64)
        for i in range(n):
            pos = origin + spacing * vin[i]
            r = sp - pos
            mag = math.sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2])
            hd = np.array([r[0] / mag, r[1] / mag, r[2] / mag])
            assert np.array_equal(bits(dirs[i]), bits(hd))
            ov, ot, _ = oracle.dda_3d(hd, shape, vin[i], spacing)
            assert cnt[i] == len(ot)
            assert np.array_equal(vox[i, :cnt[i]], ov)
            assert np.array_equal(bits(t[i, :cnt[i]]), bits(ot))


def test_quotients_past_the_double_range(oracle):
    """s / |d| overflows where (s / 2) / |d| does not: the crossings are the
    reference's own operations."""
    from conehead_amd.dda_3d_c import dda_3d_c
    for d in ([1e-308] * 3, [1e-308, -1e-308, 1.2e-308]):
        want = oracle.dda_3d(np.array(d), (9, 10, 11), (4, 5, 6), [2.0] * 3)
        got = dda_3d_c(np.array(d), (9, 10, 11), (4, 5, 6), [2.0] * 3)
        assert np.array_equal(got[0], want[0])
        assert np.array_equal(bits(got[1]), bits(want[1]))
