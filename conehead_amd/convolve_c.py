"""Drop-in for conehead's convolve_c (conehead/convolve_c.pyx:17-197).

Same signature and semantics: `dose_grid_dose` (float64, any strides) is
accumulated in place with the collapsed-cone convolution of
`dose_grid_terma`, for the cones thetas x phis (degrees) and the cumulative
kernel tables kernel.cumulative["%.2f" % phi].  The work runs on the GPU:
the FP64 TERMA is converted to FP32 on the device, the convolution runs in
the FFT form (grids whose axes fit its frames), whose FP32 result is added
into the FP64 dose on the host, or as the deterministic stencil gather,
which adds into it on the device.  Cone sets, plans, device buffers and the
pinned target of the FP32 result are kept between calls.
"""
import collections
import ctypes
import threading

import numpy as np

from . import _lib
from . import engine as _engine
from .cones import ConeSet, kernel_rows
from .device import DeviceArray, HostBuffer

_ENGINE = None
_LOCK = threading.Lock()
_CALL_LOCK = threading.Lock()   # one call at a time owns the buffers
_CONES = {}     # (thetas, phis, id(kernel)) -> (kernel rows, ConeSet)
_BUFS = collections.OrderedDict()   # grid shape -> device buffers of one
_MAX_SHAPES = 5                     # call, least recently used first
# The pinned target of FP32 results, one for all shapes: allocated per shape,
# it made a caller that goes round six shapes of 60^3 to 80 voxels pay 0.4 ms
# a call, more than the upload and download that it saves.
_PINNED = {}
_MAX_PINNED = 256 << 20             # larger results take ordinary memory


def default_engine():
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = _engine.Engine()
    return _ENGINE


def _check_grid(a, name, writable=False):
    if not isinstance(a, np.ndarray):
        a = np.asarray(a)
    if a.ndim != 3:
        raise ValueError("Buffer has wrong number of dimensions (expected 3,"
                         " got %d)" % a.ndim)
    if a.dtype != np.float64:
        raise ValueError("Buffer dtype mismatch, expected 'float64_t' but "
                         "got '%s' (%s)" % (a.dtype, name))
    if writable and not a.flags.writeable:
        raise ValueError("buffer source array is read-only (%s)" % name)
    return a


def _cones(thetas, phis, kernel):
    """The ConeSet of these angles and kernel, reused while the kernel's
    rows are unchanged (they are compared by value on every call)."""
    th = np.asarray(thetas, dtype=np.float64).ravel()
    ph = np.asarray(phis, dtype=np.float64).ravel()
    rows = kernel_rows(kernel, ph) if len(ph) else None
    key = (th.tobytes(), ph.tobytes(), id(kernel))
    with _LOCK:
        hit = _CONES.get(key)
    if hit is not None and (rows is None or np.array_equal(hit[0], rows)):
        return hit[1]
    cones = ConeSet(th, ph, kernel, semantics="convolve_c")
    with _LOCK:
        if len(_CONES) > 64:
            _CONES.clear()
        _CONES[key] = (None if rows is None else rows.copy(), cones)
    return cones


def _buffers(shape):
    with _LOCK:
        b = _BUFS.pop(shape, None)
        if b is None:
            while len(_BUFS) >= _MAX_SHAPES:
                _BUFS.popitem(last=False)
            b = {"t64": DeviceArray(shape, np.float64),
                 "t": DeviceArray(shape, np.float32),
                 "part": DeviceArray(shape, np.float32),
                 "box": DeviceArray((6,), np.int32)}
        _BUFS[shape] = b
        return b


def _host_result(shape):
    """A float32 array of this shape for the result: a view of the pinned
    target, or ordinary memory where that cannot hold it."""
    nbytes = 4 * int(np.prod(shape))
    if nbytes > _MAX_PINNED:
        return np.empty(shape, np.float32)
    buf = _PINNED.get("buf")
    if buf is None or buf.nbytes < nbytes:
        _PINNED.clear()
        try:
            buf = _PINNED["buf"] = HostBuffer(nbytes)
        except _lib.CHError:
            return np.empty(shape, np.float32)
    return np.ctypeslib.as_array(ctypes.cast(buf.ptr, _lib.c_f32p), shape)


def _add(dose, part):
    """dose += part, `part` a C-ordered float32 array.

    numpy adds along the dose's layout, which costs a cache line of the
    result per element where the dose's fastest axis is not the last one (a
    Fortran-ordered dose of 128^3 voxels: 27 ms); those go in tiles."""
    if dose.flags.aligned and dose.size:
        L = _lib.lib()
        if dose.flags.c_contiguous:
            _lib.check(L.ch_host_add_f32(dose.ctypes.data, part.ctypes.data,
                                         dose.size))
            return
        # axes from the largest step to the smallest, those of one element
        # first; next to each other only if they do not overlap
        order = sorted(range(3), key=lambda a: (
            dose.shape[a] > 1, -abs(dose.strides[a])))
        steps = [(abs(dose.strides[a]), dose.shape[a]) for a in order]
        apart = all(s[0] >= t[0] * t[1]
                    for s, t in zip(steps, steps[1:] + [(8, 1)])
                    if s[1] > 1)
        if order[2] != 2 and apart and \
                all(s % 8 == 0 for s in dose.strides):
            axes = ([a for a in range(3) if a not in (order[2], 2)] +
                    [order[2], 2])
            i64 = ctypes.c_int64 * 3
            _lib.check(L.ch_host_add_f32_strided(
                dose.ctypes.data, part.ctypes.data,
                i64(*[dose.shape[a] for a in axes]),
                i64(*[dose.strides[a] // 8 for a in axes]),
                i64(*[part.strides[a] // 4 for a in axes])))
            return
    np.add(dose, part, out=dose)


def _convert(dst, src):
    types = {np.dtype(np.float32): _lib.CH_F32,
             np.dtype(np.float64): _lib.CH_F64}
    _lib.check(_lib.lib().ch_convert(dst.ptr, types[dst.dtype], src.ptr,
                                     types[src.dtype], dst.size, 0, None))


def convolve_c(dose_grid_terma, dose_grid_dose, dose_grid_dim, thetas, phis,
               kernel, method="auto"):
    """Accumulate the cone convolution of TERMA into `dose_grid_dose`.

    method: "auto" (the FFT form where the grid fits its frames, else the
    gather), "fft" or "gather"."""
    terma = _check_grid(dose_grid_terma, "dose_grid_terma")
    dose = _check_grid(dose_grid_dose, "dose_grid_dose", writable=True)
    if dose.shape != terma.shape:
        # the reference indexes dose with the TERMA grid's voxel indices
        raise ValueError("dose grid %s does not match TERMA grid %s" %
                         (dose.shape, terma.shape))
    if method not in ("auto", "fft", "gather"):
        raise ValueError("method must be auto, fft or gather")
    dims = np.asarray(dose_grid_dim, dtype=np.float64).reshape(3)
    cones = _cones(thetas, phis, kernel)
    if cones.n_cones == 0:
        return None
    from .batch import spectral_ok
    shape = tuple(int(v) for v in terma.shape)
    fft = method == "fft" or (method == "auto" and spectral_ok(shape))
    eng = default_engine()
    plan = eng.plan(shape, dims, cones)
    with _CALL_LOCK:
        _run(plan, shape, terma, dose, fft)
    return None


def _run(plan, shape, terma, dose, fft):
    b = _buffers(shape)
    b["t64"].upload(np.ascontiguousarray(terma))
    _convert(b["t"], b["t64"])
    if fft:
        # the FP32 result crosses the bus once, into pinned memory, instead
        # of the FP64 dose there and back (101 x 97 x 83 voxels: a download
        # of the dose 0.47 ms and its upload 0.18 ms of the call's 0.94)
        plan.spectrum()
        _engine.convolve_fft(plan, b["t"], b["part"])
        part = _host_result(shape)
        b["part"].download(out=part)
        _add(dose, part)
        return
    if "dose" not in b:
        b["dose"] = DeviceArray(shape, np.float64)
    b["dose"].upload(np.ascontiguousarray(dose))
    _engine.support_box(b["t"], shape, b["box"])
    _engine.convolve_f64(plan, b["t"], b["dose"], b["box"])
    if dose.flags.c_contiguous:
        b["dose"].download(out=dose)
    else:
        np.copyto(dose, b["dose"].download())
