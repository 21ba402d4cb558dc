"""Conehead.calculate on the GPU engine (drop-in for conehead/conehead.py:520).

The reference's flow -- density interpolation, hit test, effective depth,
off-axis distance, fluence, softening and horn, TERMA, polyenergetic kernel,
dose (conehead/conehead.py:522-773) -- runs as one fused TERMA launch and
the collapsed-cone convolution (five FFT passes, or one gather launch),
with every intermediate kept in HBM.  The
dose is returned and stored in self.dose_grid.dose (the reference plots it
and discards it).

Settings keys are the reference's (example.py:27-58).  Optional keys:
  thetas, phis, kernel -- the cone set handed to the convolution (default:
      12 azimuths and all 48 polar keys of PolyenergeticKernel, the cone set
      of the reference's convolve_c call, conehead/conehead.py:780-794);
  semantics -- "convolve_c" (default), "cuda_dose" (y-polar cones and the
      index arithmetic of conehead/conehead.py:385-488; `kernel` is then a
      [n_phi, >=5996] cumulative table and `phis` its angles; without them
      the reference's live call: the EDKnrc KernelPoly of
      settings['energy_weights'], its 48 polar angles and 12 float32
      azimuths, conehead/conehead.py:686-738) or "physics"
      (the cuda_dose cones aligned with the beam and the kernel looked up at
      the radiological distance through the densities; without `kernel` the
      EDKnrc polyenergetic kernel of settings['energy_weights'] merged into
      settings.get('n_phi', 12) polar groups);
  convolution -- "fft" (default for the convolve_c and cuda_dose
      semantics: the cone stencil summed into one kernel and applied with
      zero-padded FFTs, ch_convolve_fft) or "gather" (the direct stencil
      sum, ch_convolve); physics mode always gathers, since its kernel
      distance depends on the densities along each path;
  density_xy_swap -- True (default) reproduces the reference's density
      resampling, whose meshgrid(indexing='xy') evaluation at the grid nodes
      swaps the x and y axes (conehead/conehead.py:562-567); False uses the
      densities as given.
"""
import collections
import threading

import numpy as np

from . import engine as _engine
from .cones import ConeSet, beam_frame, default_thetas, kernel_phis
from .batch import DevicePool, spectral_ok
from .device import HostPool, Stream
from .dosegrid import DoseGrid
from .kernel import EdkSet, merge_polar
from .kernel2 import PolyenergeticKernel
from .phantom import CtPhantom

# The packaged kernel table, parsed once, and the cone sets of it most
# recently asked for, by the values of their angles.  A whole call of 50^3
# voxels and 576 cones spent 3.0 of its 3.6 ms on parsing the table, building
# the cones and hashing their rows.
_DEFAULT_LOCK = threading.Lock()
_DEFAULT = {"kernel": None, "cones": collections.OrderedDict()}


def _default_cones(thetas, phis):
    """ConeSet of the packaged kernel (phis None: all its polar angles)."""
    with _DEFAULT_LOCK:
        if _DEFAULT["kernel"] is None:
            _DEFAULT["kernel"] = PolyenergeticKernel()
        kernel, sets = _DEFAULT["kernel"], _DEFAULT["cones"]
        th = np.array(thetas, dtype=np.float64).ravel()
        ph = np.array(kernel_phis(kernel) if phis is None else phis,
                      dtype=np.float64).ravel()
        key = (th.tobytes(), ph.tobytes())
        cones = sets.pop(key, None)
        if cones is None:
            cones = ConeSet(th, ph, kernel)
        sets[key] = cones
        while len(sets) > 8:
            sets.popitem(last=False)
        return cones


def dose_grid_densities(phantom, swap_xy=True):
    """Densities on the dose grid (the phantom's own grid).

    The reference interpolates the phantom linearly at the nodes
    linspace(origin, origin + n*s, n) of the same axes it interpolates on,
    so every value is a node value; its meshgrid uses indexing='xy', which
    lays the result out as [y][x][z]."""
    d = np.asarray(phantom.densities, dtype=np.float32)
    if not swap_xy:
        return np.ascontiguousarray(d)
    if d.shape[0] != d.shape[1]:
        raise ValueError(
            "the reference's xy-swapped density resampling is only defined "
            "for phantoms with size[0] == size[1]; pass "
            "settings['density_xy_swap'] = False")
    return np.ascontiguousarray(d.transpose(1, 0, 2))


class Conehead:

    def __init__(self, engine=None):
        self._engine = engine
        self._stream = None
        self._pools = None
        self.dose_grid = None

    @property
    def stream(self):
        """The instance's stream, kept across calls so its TERMA flag, FFT
        work grids and gather workspace are allocated once."""
        if self._stream is None:
            self._stream = Stream()
        return self._stream

    def _pool_pair(self):
        """(device grids, pinned results) kept between calls: an allocation
        of each grid cost 0.17 ms, a download into fresh pageable memory ran
        at a quarter of the link.  Results view pinned buffers, which return
        to the pool when their last array is gone.  A caller that keeps its
        results gets ordinary memory once the pinned ones alive and idle
        would pass max_bytes."""
        if self._pools is None:
            self._pools = (DevicePool(max_free_bytes=1 << 30),
                           HostPool(max_free_bytes=512 << 20,
                                    max_bytes=1 << 30))
        return self._pools

    def close(self):
        """Frees the device grids and pinned buffers kept between calls (not
        the results handed out: their memory goes with their last view).  A
        later calculate() keeps its own again."""
        if self._pools is not None:
            for pool in self._pools:
                pool.close()
            self._pools = None

    @property
    def engine(self):
        if self._engine is None:
            from .convolve_c import default_engine
            self._engine = default_engine()
        return self._engine

    def calculate(self, source, block, phantom, settings):
        """TERMA and dose of one beam; returns the FP32 dose grid.

        The returned arrays are the caller's, as numpy's are.  Up to 1 GiB of
        results still referenced they lie in pinned memory, which goes to a
        later call when the last view of them is dropped; results past that
        lie in ordinary memory.

        The dose grid is the phantom's own (conehead/conehead.py:536) unless
        settings['dose_grid'] = (size, origin, spacing) names another one;
        the densities are then resampled on the GPU (ch_resample_linear)
        with the reference's interpolation and layout.  A CtPhantom's
        densities are made on the GPU from its CT numbers
        (ch_ct_to_density) and resampled there."""
        eng = self.engine
        swap = settings.get("density_xy_swap", True)
        grid = settings.get("dose_grid")
        s = self.stream
        grids, pinned = self._pool_pair()
        held = []                   # back to the pool once the stream is idle

        def device(shape, dtype=np.float32):
            held.append(grids.get(tuple(shape), np.dtype(dtype)))
            return held[-1]

        def upload(arr):
            a = np.ascontiguousarray(arr)
            return device(a.shape, a.dtype).upload(a, s)

        d_dens = None
        on_device = hasattr(phantom, "device_densities")  # CtPhantom
        if grid is None and not on_device:
            self.dose_grid = DoseGrid(phantom.size, phantom.origin,
                                      phantom.spacing)
            dens = dose_grid_densities(phantom, swap)
            dens_shape = dens.shape
            d_rho = upload(dens)
        else:
            # resampling the phantom's own grid onto itself gives every
            # node's value, i.e. dose_grid_densities bit for bit
            from .density import ct_to_density, resample
            self.dose_grid = DoseGrid(*grid) if grid is not None else \
                DoseGrid(phantom.size, phantom.origin, phantom.spacing)
            if type(phantom) is CtPhantom:
                d_src = ct_to_density(
                    upload(phantom.ct), phantom.curve,
                    None if phantom.labels is None
                    else upload(phantom.labels), phantom.overrides,
                    device(phantom.ct.shape), stream=s)
            elif on_device:
                d_src = phantom.device_densities(stream=s)
            else:
                d_src = upload(phantom.densities)
            d_rho = d_dens = resample(
                d_src, tuple(phantom.size), phantom.origin, phantom.spacing,
                self.dose_grid.size, self.dose_grid.origin,
                self.dose_grid.spacing, swap_xy=swap,
                d_dst=device(int(v) for v in self.dose_grid.size), stream=s)
            dens_shape = d_rho.shape
        shape = tuple(int(v) for v in self.dose_grid.size)
        origin = np.asarray(self.dose_grid.origin, dtype=np.float64)
        spacing = np.asarray(self.dose_grid.spacing, dtype=np.float64)
        if dens_shape != shape:
            raise ValueError("densities %s do not match size %s" %
                             (dens_shape, shape))

        semantics = settings.get("semantics", "convolve_c")
        kernel = settings.get("kernel")
        physics = semantics == "physics"
        default = semantics == "convolve_c" and kernel is None
        if default:
            phis = settings.get("phis")
        elif semantics == "convolve_c":
            phis = settings.get("phis")
            phis = kernel_phis(kernel) if phis is None else phis
        elif physics and kernel is None:
            # EDKnrc polyenergetic kernel of the beam's spectrum
            # (conehead/conehead.py:686-704), merged into polar groups
            poly = EdkSet.load().poly(settings["energy_weights"])
            phis, kernel = merge_polar(poly.angles, poly.kernel_cum,
                                       int(settings.get("n_phi", 12)))
        elif semantics == "cuda_dose" and kernel is None:
            # the reference's live dose call (conehead/conehead.py:686-738):
            # KernelPoly of settings['energy_weights'] (48 x 5996), its 48
            # float32 polar angles and 12 float32 azimuths 0, 30, ..., 330
            if settings.get("phis") is not None:
                raise ValueError("cuda_dose semantics: settings['phis'] "
                                 "needs settings['kernel'] too")
            poly = EdkSet.load().poly(settings["energy_weights"])
            kernel = poly.kernel_cum
            phis = np.asarray(poly.angles)
        else:
            if kernel is None or settings.get("phis") is None:
                raise ValueError("%s semantics needs settings['kernel'] "
                                 "(cumulative table) and settings['phis']"
                                 % semantics)
            phis = settings["phis"]
        thetas = settings.get("thetas")
        if thetas is None:
            thetas = (np.linspace(0, 360 - 360 / 12, 12, dtype=np.float32)
                      if semantics == "cuda_dose" else default_thetas(12))
        cones = _default_cones(thetas, phis) if default else \
            ConeSet(thetas, phis, kernel, semantics=semantics,
                    frame=beam_frame(source) if physics else None)

        method = settings.get("convolution", "fft")
        if method not in ("fft", "gather"):
            raise ValueError("settings['convolution'] must be 'fft' or "
                             "'gather'")
        # the FFT form takes axes of up to 512 voxels; beyond, the gather
        use_fft = method == "fft" and not physics and spectral_ok(shape)
        d_terma = device(shape)
        # the support box only serves the gathers, which clip to it
        d_box = None if use_fft else device((6,), np.int32)
        d_raster = eng.aperture(block, s)
        beam = _engine.beam_struct(source, settings, d_raster, d_rho,
                                   d_terma, d_box)
        # queued without a wait in between; the geometry flag is read once
        # at the end, and first where something else fails
        _engine.terma([beam], shape, origin, spacing, stream=s, check=False)
        results = []
        try:
            plan = eng.plan(shape, spacing, cones)
            d_dose = device(shape)
            if physics:
                _engine.convolve_rad(plan, d_terma, d_rho, d_dose, d_box,
                                     stream=s)
            elif use_fft:
                _engine.convolve_fft(plan, d_terma, d_dose, stream=s)
            else:
                _engine.convolve(plan, d_terma, d_dose, d_box, stream=s)
            for d in (d_dose, d_terma, d_dens):
                if d is not None:
                    results.append((d, pinned.try_get(d.nbytes)))
                    if results[-1][1] is not None:
                        d.download_async(results[-1][1], stream=s)
            s.sync()
        except Exception:
            s.sync()
            _engine.terma_check(s)
            raise
        try:
            _engine.terma_check(s)
        except Exception:
            for _, h in results:
                if h is not None:
                    pinned.put(h)
            raise
        arrays = [d.download(stream=s) if h is None
                  else pinned.as_array(h, shape) for d, h in results]
        for d in held:
            grids.put(d)
        self.dose_grid_terma = arrays[1]
        self.dose_grid_densities = dens if d_dens is None else arrays[2]
        self.dose_grid.dose = arrays[0]
        return arrays[0]
