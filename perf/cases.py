"""Timed cases of the dose engine: what its users have it compute, through
the package's public entry points.

Kinds of case:
  calculate  Conehead.calculate, host densities (or CT numbers with a label
             map) to host dose and TERMA: the reference's own call;
  dropin     convolve_c on host float64 arrays, accumulated in place;
  beam       one beam on device buffers: TERMA, then the FFT convolution,
             queued call by call or replayed as one captured graph;
  batch      BatchEngine on uneven phantoms, one dose grid per beam;
  replay     BatchGraph: many MLC beams on one phantom, captured once;
  physics    the convolution with radiological kernel distances;
  gather     the direct stencil gather (grids with an axis beyond the FFT
             form's 512 voxels always take it);
  density    CT numbers to densities, resampled onto a dose grid.

Grids of 40 to 200 voxels per axis and voxels of 2 to 5 mm are what a plan
uses; 50 voxels of 4 mm is the reference's example, 128 of 2.5 mm the
benchmark's beam, 64 to 200 odd and uneven its batch.
"""
import itertools
import math
import os

import numpy as np
import torch

SETTINGS = {
    "sPri": 0.90924, "sAnn": 2.887e-3, "zAnn": 4.0, "rInner": 0.2,
    "rOuter": 1.4, "zExp": 12.5, "sExp": 8.289e-3, "kExp": 0.4816,
    "softRatio": 0.0025, "softLimit": 20, "hornRatio": 0.0065,
    "fluenceResampling": 3,
    "energy_weights": {
        "0.5": 0.08196, "1.0": 0.12385, "1.5": 0.10605, "2.0": 0.08307,
        "2.5": 0.05881, "3.0": 0.03911, "3.5": 0.02131, "4.0": 0.02426,
        "4.5": 0.0, "5.0": 0.00881, "5.5": 0.0, "6.0": 0.00498,
    },
}
# mass attenuation of water (MeV, cm^2/g), linear in between
WATER = ((0.5, 9.687e-2), (1.0, 7.072e-2), (1.5, 5.754e-2), (2.0, 4.942e-2),
         (3.0, 3.969e-2), (4.0, 3.403e-2), (5.0, 3.031e-2), (6.0, 2.770e-2))
CT_CURVE = ((-1000.0, 0.0012), (-500.0, 0.5), (0.0, 1.0), (300.0, 1.16),
            (1500.0, 1.82), (3000.0, 2.9))
CT_OVERRIDES = {3: 1.0, 7: 0.26}


def listed():
    return [
        # the reference's example: one call, host to host, its default
        # kernel (48 polar angles) and azimuths; latency and host work
        {"name": "calculate_example", "kind": "calculate", "x": 50, "y": 50,
         "z": 50, "mm": 4.0, "gantry": 0.0, "side": 10.0, "n_phi": 48},
        # a patient beam: CT numbers with structures, resampled onto the
        # dose grid, an oblique beam
        {"name": "calculate_ct", "kind": "calculate", "x": 97, "y": 97,
         "z": 84, "mm": 3.0, "gantry": 35.0, "side": 12.0, "n_phi": 12,
         "ct": 1.5},
        # callers of the reference's convolution, float64 on the host
        {"name": "dropin_odd", "kind": "dropin", "x": 101, "y": 97, "z": 83,
         "mm": 2.5, "gantry": 0.0, "side": 8.0, "n_phi": 8},
        # the smallest device-resident beam: launches count
        {"name": "beam_small", "kind": "beam", "x": 40, "y": 40, "z": 40,
         "mm": 5.0, "gantry": 0.0, "side": 6.0, "n_phi": 8, "graph": False},
        # the benchmark's heterogeneous beam, replayed
        {"name": "beam_128", "kind": "beam", "x": 128, "y": 128, "z": 128,
         "mm": 2.5, "gantry": 0.0, "side": 10.0, "n_phi": 12, "graph": True},
        # a ragged grid, an MLC aperture and an oblique beam
        {"name": "beam_odd_mlc", "kind": "beam", "x": 173, "y": 97, "z": 141,
         "mm": 2.2, "gantry": 207.5, "side": 0.0, "n_phi": 8,
         "graph": False},
        # the largest grid of the uneven workload, the y-polar cones
        {"name": "beam_large", "kind": "beam", "x": 200, "y": 200, "z": 160,
         "mm": 2.0, "gantry": 120.0, "side": 15.0, "n_phi": 12,
         "graph": True, "semantics": "cuda_dose"},
        # requests of different grids, beam counts and cone sets, doses
        # left on the device for the next consumer
        {"name": "batch_uneven", "kind": "batch", "requests": 6, "mix": 11},
        # the beams of a plan, optimised over and over: captured once
        {"name": "replay_mlc", "kind": "replay", "x": 128, "y": 128,
         "z": 128, "mm": 2.5, "n_phi": 8, "beams": 24},
        # kernel distances through the densities
        {"name": "physics_96", "kind": "physics", "x": 96, "y": 96, "z": 96,
         "mm": 3.0, "gantry": 20.0, "side": 10.0, "n_phi": 12},
        # a long phantom: beyond the FFT form's frames
        {"name": "gather_long", "kind": "gather", "x": 64, "y": 56,
         "z": 560, "mm": 2.5, "gantry": 0.0, "side": 12.0, "n_phi": 8},
        # a whole CT series onto the dose grid
        {"name": "density_series", "kind": "density", "x": 512, "y": 512,
         "z": 120, "mm": 0.98, "n": 160, "nz": 128, "dose_mm": 2.5},
    ]


def draw(rng):
    """One more case of the same ranges (sizes over their logarithm)."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("calculate", "dropin", "beam", "beam", "beam",
                       "batch", "replay", "physics", "gather", "density"))
    mm = round(rng.uniform(2.0, 5.0), 2)
    gantry = round(rng.uniform(0.0, 359.0), 1)
    side = round(rng.uniform(4.0, 15.0), 1)
    n_phi = rng.choice((4, 6, 8, 12))
    if kind == "calculate":
        n = size(40, 128)
        case = {"x": n, "y": n, "z": size(40, 128), "mm": mm,
                "gantry": gantry, "side": side, "n_phi": n_phi}
        if rng.random() < 0.5:
            case["ct"] = round(rng.uniform(1.5, 2.5), 2)
    elif kind == "dropin":
        case = {"x": size(40, 128), "y": size(40, 128), "z": size(40, 128),
                "mm": mm, "gantry": gantry, "side": side, "n_phi": n_phi}
    elif kind == "beam":
        case = {"x": size(40, 200), "y": size(40, 200), "z": size(40, 160),
                "mm": mm, "gantry": gantry,
                "side": side if rng.random() < 0.6 else 0.0, "n_phi": n_phi,
                "graph": rng.random() < 0.5}
        if rng.random() < 0.3:
            case["semantics"] = "cuda_dose"
    elif kind == "batch":
        case = {"requests": rng.randint(2, 6), "mix": rng.randint(20, 9999)}
    elif kind == "replay":
        case = {"x": size(48, 128), "y": size(48, 128), "z": size(48, 128),
                "mm": mm, "n_phi": n_phi, "beams": size(2, 24)}
    elif kind == "physics":
        case = {"x": size(40, 96), "y": size(40, 96), "z": size(40, 96),
                "mm": mm, "gantry": gantry, "side": side, "n_phi": n_phi}
    elif kind == "gather":
        case = {"x": size(40, 64), "y": size(40, 64), "z": size(64, 560),
                "mm": mm, "gantry": gantry, "side": side, "n_phi": n_phi}
    else:
        case = {"x": size(128, 512), "y": size(128, 512), "z": size(40, 120),
                "mm": round(rng.uniform(0.9, 2.0), 2), "n": size(64, 160),
                "nz": size(64, 128), "dose_mm": mm}
    return dict(case, kind=kind)


# ---------------------------------------------------------------- inputs --

def shape_of(case):
    return case["x"], case["y"], case["z"]


def grid_of(shape, mm):
    """Origin and spacing in cm, isocentre at the middle, as float32 holds
    them (the phantoms keep float32)."""
    sp = float(np.float32(mm / 10.0))
    org = [float(np.float32(-(n - 1) / 2.0 * sp)) for n in shape]
    return np.array(org), np.array([sp] * 3)


def ellipsoids(shape, rng, n):
    ax = np.ogrid[:shape[0], :shape[1], :shape[2]]
    for _ in range(n):
        c = rng.uniform(0.25, 0.75, 3) * shape
        r = rng.uniform(0.08, 0.25, 3) * shape
        yield sum(((ax[a] - c[a]) / r[a]).astype(np.float32) ** 2
                  for a in range(3)) <= 1.0


def densities_of(shape, seed):
    """Water with lungs, bones and noise."""
    rng = np.random.default_rng([seed, 1])
    rho = np.ones(shape, np.float32)
    for k, m in enumerate(ellipsoids(shape, rng, 4)):
        rho[m] = rng.uniform(0.2, 0.35) if k < 2 else rng.uniform(1.5, 1.9)
    rho += np.float32(0.02) * rng.standard_normal(shape, dtype=np.float32)
    return np.clip(rho, 0.0, None)


def ct_of(shape, seed):
    """CT numbers: air around a body with lungs and bones, scanner noise;
    and a structure map."""
    rng = np.random.default_rng([seed, 2])
    ct = np.full(shape, -1000, np.int16)
    ax = np.ogrid[:shape[0], :shape[1], :shape[2]]
    body = sum(((ax[a] - shape[a] / 2) / (0.45 * shape[a])).astype(
        np.float32) ** 2 for a in range(2)) <= 1.0
    ct[np.broadcast_to(body, shape)] = 0
    labels = np.zeros(shape, np.uint8)
    for k, m in enumerate(ellipsoids(shape, rng, 4)):
        ct[m] = rng.integers(-850, -600) if k < 2 else \
            rng.integers(300, 1400)
        labels[m] = (0, 7, 0, 3)[k]
    ct += rng.integers(-25, 26, size=shape, dtype=np.int16)
    return ct, labels


def mlc_of(rng):
    """Leaf bank (mm): 60 pairs of 5 mm leaves, openings of 20-200 mm."""
    bound = -150.0 + 5.0 * np.arange(61)
    width, centre = rng.uniform(20.0, 200.0), rng.uniform(-20.0, 20.0)
    wob = rng.uniform(-0.15, 0.15, 60) * width
    jy = rng.uniform(10.0, 100.0)
    return (bound, centre - width / 2.0 + wob, centre + width / 2.0 + wob,
            (-120.0, 120.0), (-jy, jy))


def aperture_of(side, rng):
    return ("square", side) if side > 0 else ("mlc",) + mlc_of(rng)


def requests_of(case):
    """The uneven batch: per request shape, voxel size, polar angles and
    the beams' gantry angles and field sides."""
    rng = np.random.default_rng([case["mix"], 3])
    out = []
    for _ in range(case["requests"]):
        shape = (int(rng.integers(64, 161)), int(rng.integers(64, 161)),
                 int(rng.integers(64, 141)))
        beams = [(round(float(rng.uniform(0, 359)), 2),
                  round(float(rng.uniform(4, 15)), 2))
                 for _ in range(int(rng.integers(1, 6)))]
        out.append((shape, round(float(rng.uniform(2, 5)), 2),
                    int(rng.choice((4, 6, 8, 12))), beams))
    return out


def field_terma(shape, org, sp, gantry, side, seed):
    """A beam-shaped TERMA grid (float32, on the GPU): zero outside the
    divergent field, attenuated and noisy inside it."""
    pos, vy, tr = geometry(gantry)
    p = [torch.arange(shape[a], dtype=torch.float64, device="cuda")
         .mul(sp[a]).add(org[a]).reshape([-1 if a == b else 1
                                          for b in range(3)])
         for a in range(3)]
    depth = sum(vy[a] * (p[a] - pos[a]) for a in range(3))
    q0 = sum(tr[0, a] * (p[a] - pos[a]) for a in range(3)) * 100.0 / depth
    q2 = sum(tr[2, a] * (p[a] - pos[a]) for a in range(3)) * 100.0 / depth
    lit = (q0.abs() < side / 2) & (q2.abs() < side / 2)
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    t = torch.exp(-0.05 * (depth - 80.0)) * (100.0 / depth) ** 2 * \
        (1.0 + 0.02 * torch.randn(shape, generator=g, device="cuda",
                                  dtype=torch.float64))
    return torch.where(lit, t, torch.zeros_like(t)).float().contiguous()


def cone_table(n_phi):
    """(angles, cumulative rows) of the package's 6 MV kernel data: the 48
    polar bins merged into n_phi groups (48: as they are)."""
    import conehead_amd
    path = os.path.join(os.path.dirname(conehead_amd.__file__), "data",
                        "varian_6.csv")
    tab = np.loadtxt(path, delimiter=",", skiprows=1)
    radii = np.linspace(0.05, 60.0, 5996)
    angles = sorted(set(180 - a for a in tab[:, 0]))
    rows = []
    for a in angles:
        m = np.abs((180 - tab[:, 0]) - a) < 1e-9
        rows.append(np.interp(radii, tab[m, 1],
                              np.cumsum(tab[m, 2] / 0.289622754141)))
    rows = np.stack(rows)
    if n_phi == 48:
        return np.array(angles), rows
    w = 48 // n_phi
    phis = [angles[g * w] + (angles[1] - angles[0]) * w / 2.0
            for g in range(n_phi)]
    return np.array(phis), rows.reshape(n_phi, w, -1).sum(axis=1)


# ------------------------------------------------------- a user's program --

_KEPT = {}


def program():
    """What a program keeps: the engine with its plans, the batch engine,
    its stream, and the cone sets (their kernel tables are read once)."""
    if not _KEPT:
        from conehead_amd.batch import BatchEngine
        from conehead_amd.convolve_c import default_engine
        from conehead_amd.device import Stream
        _KEPT["engine"] = default_engine()
        _KEPT["batch"] = BatchEngine(engine=_KEPT["engine"])
        _KEPT["stream"] = Stream()
        _KEPT["cones"] = {}
        _KEPT["keys"] = itertools.count()
    return _KEPT


def tables(n_phi):
    kept = program()
    if n_phi not in kept["cones"]:
        kept["cones"][n_phi] = cone_table(n_phi)
    return kept["cones"][n_phi]


def kernel_dict(n_phi):
    from conehead_amd.kernel2 import ConeKernel
    phis, rows = tables(n_phi)
    return phis, ConeKernel({"%.2f" % p: r for p, r in zip(phis, rows)})


def cone_set(n_phi, semantics="convolve_c", source=None):
    from conehead_amd.cones import ConeSet, beam_frame, default_thetas
    kept = program()
    key = (n_phi, semantics)
    if source is None and key in kept["cones"]:
        return kept["cones"][key]
    if semantics == "convolve_c":
        phis, kernel = kernel_dict(n_phi)
    else:
        phis, rows = tables(n_phi)
        phis, kernel = 180.0 - phis, rows
    cones = ConeSet(default_thetas(12), phis, kernel, semantics=semantics,
                    frame=None if source is None else beam_frame(source))
    if source is None:
        kept["cones"][key] = cones
    return cones


def source_of(gantry):
    from conehead_amd.source import Source
    s = Source("varian_clinac_6MV")
    s.gantry = gantry
    return s


def block_of(aperture):
    from conehead_amd.block import Block
    b = Block()
    if aperture[0] == "square":
        b.set_square(aperture[1])
    else:
        b.set_mlc(*aperture[1:])
    return b


class _Memory:
    """A DeviceArray's memory as torch takes it."""

    def __init__(self, d):
        self.owner = d
        self.__cuda_array_interface__ = {
            "shape": d.shape, "typestr": d.dtype.str,
            "data": (d.ptr, False), "version": 2}


def view(d):
    return torch.as_tensor(_Memory(d), device="cuda")


class State(dict):
    """A prepared case; what it holds is closed, in order, when dropped."""

    def __del__(self):
        for close, args in self.get("close", ()):
            close(*args)


def to_device(a, stream):
    from conehead_amd.device import DeviceArray
    if isinstance(a, torch.Tensor):
        a = a.cpu().numpy()
    return DeviceArray.from_host(a, stream=stream)


def prepare(case, seed):
    return globals()["prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["run_" + state["kind"]](state)


def prepare_calculate(case, seed):
    from conehead_amd.conehead import Conehead
    from conehead_amd.phantom import CtPhantom, Phantom
    program()
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    st = dict(SETTINGS)
    if case["n_phi"] != 48:
        st["phis"], st["kernel"] = kernel_dict(case["n_phi"])
    if case.get("ct"):
        cshape, corg, csp = ct_grid(case)
        ct, labels = ct_of(cshape, seed)
        phantom = CtPhantom(ct, corg, csp, curve=CT_CURVE, labels=labels,
                            overrides=CT_OVERRIDES)
        st["dose_grid"] = (list(shape), org, sp)
    else:
        phantom = Phantom(densities_of(shape, seed), org, sp)
    return State(kind="calculate", conehead=Conehead(), phantom=phantom,
                 source=source_of(case["gantry"]),
                 block=block_of(("square", case["side"])), settings=st)


def run_calculate(s):
    c = s["conehead"]
    dose = c.calculate(s["source"], s["block"], s["phantom"], s["settings"])
    return {"dose": dose, "terma": c.dose_grid_terma}


def ct_grid(case):
    """The CT series around a dose grid: finer voxels, a little larger."""
    mm = case["ct"]
    n = [int(1.1 * case[a] * case["mm"] / mm) for a in "xyz"]
    return (tuple(n),) + grid_of(n, mm)


def dropin_inputs(case, seed):
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    t = field_terma(shape, org, sp, case["gantry"], case["side"], seed)
    rng = np.random.default_rng([seed, 4])
    return (t.double().cpu().numpy(), rng.random(shape) * 0.1, sp)


def prepare_dropin(case, seed):
    from conehead_amd.cones import default_thetas
    terma, dose, sp = dropin_inputs(case, seed)
    phis, kernel = kernel_dict(case["n_phi"])
    return State(kind="dropin", terma=terma, dose=dose, dims=sp,
                 thetas=default_thetas(12), phis=phis, kernel=kernel)


def run_dropin(s):
    from conehead_amd.convolve_c import convolve_c
    convolve_c(s["terma"], s["dose"], s["dims"], s["thetas"], s["phis"],
               s["kernel"])
    return s["dose"]


def prepare_beam(case, seed):
    from conehead_amd import engine as E
    from conehead_amd.device import DeviceArray, Stream
    eng, stream = program()["engine"], program()["stream"]
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    cones = cone_set(case["n_phi"], case.get("semantics", "convolve_c"))
    rho = to_device(densities_of(shape, seed), stream)
    terma, dose = DeviceArray(shape), DeviceArray(shape)
    ap = eng.aperture(block_of(aperture_of(
        case["side"], np.random.default_rng([seed, 5]))), stream)
    beam = E.beam_struct(source_of(case["gantry"]), SETTINGS, ap, rho, terma,
                         None)
    plan = eng.plan(shape, sp, cones)
    plan.spectrum(stream)
    s = State(kind="beam", E=E, beam=beam, shape=shape, org=org, sp=sp,
              plan=plan, terma=terma, dose=dose, stream=stream, graph=None,
              out={"dose": view(dose), "terma": view(terma)})
    if case["graph"]:
        # captured on a stream of its own, whose scratch the graph holds
        s["stream"] = own = Stream()
        run_beam(s)
        own.sync()
        with E.Graph.capture(own) as cap:
            run_beam(s)
        s.update(graph=cap.graph, stream=stream, own=own,
                 close=((stream.sync, ()), (cap.graph.close, ())))
    return s


def run_beam(s):
    if s["graph"] is not None:
        s["graph"].launch(s["stream"])
        return s["out"]
    E = s["E"]
    E.terma([s["beam"]], s["shape"], s["org"], s["sp"], stream=s["stream"],
            check=False)
    E.convolve_fft(s["plan"], s["terma"], s["dose"], stream=s["stream"])
    return s["out"]


def prepare_batch(case, seed):
    from conehead_amd.batch import DoseRequest
    kept = program()
    reqs = []
    for i, (shape, mm, n_phi, beams) in enumerate(requests_of(case)):
        org, sp = grid_of(shape, mm)
        reqs.append(DoseRequest(
            densities_of(shape, seed + 1000 * i), org, sp,
            [(source_of(g), block_of(("square", a)), SETTINGS)
             for g, a in beams], cone_set(n_phi),
            key="phantom %d" % next(kept["keys"])))
    be, stream = kept["batch"], kept["stream"]
    outs = []
    s = State(kind="batch", engine=be, requests=reqs, stream=stream,
              outs=outs, views={}, close=((stream.sync, ()),
                                          (be.release, (outs,))) +
              tuple((be.evict, (r.key,)) for r in reqs))
    for r in reqs:        # the phantoms are resident, the plans built
        be.densities(r, stream)
        be.engine.plan(r.shape, r.spacing, r.cones).spectrum(stream)
    return s


def run_batch(s):
    be, views = s["engine"], s["views"]
    be.release(s["outs"])
    s["outs"][:] = be.collect(be.launch(s["requests"], s["stream"]),
                              download=False)
    got = []
    for outs in s["outs"]:
        for d in outs:
            if (d.ptr, d.shape) not in views:
                views[d.ptr, d.shape] = view(d)
            got.append(views[d.ptr, d.shape])
    return got


def replay_beams(case, seed):
    rng = np.random.default_rng([seed, 6])
    return [(round(float(rng.uniform(0, 359)), 2), ("mlc",) + mlc_of(rng))
            for _ in range(case["beams"])]


def prepare_replay(case, seed):
    from conehead_amd.batch import BatchGraph, DoseRequest
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    req = DoseRequest(densities_of(shape, seed), org, sp,
                      [(source_of(g), block_of(a), SETTINGS)
                       for g, a in replay_beams(case, seed)],
                      cone_set(case["n_phi"]))
    graph = BatchGraph([req], engine=program()["engine"])
    return State(kind="replay", graph=graph, close=((graph.close, ()),),
                 out=[view(d) for d in graph.outs[0]])


def run_replay(s):
    s["graph"].launch()
    return s["out"]


def prepare_physics(case, seed):
    from conehead_amd import engine as E
    from conehead_amd.device import DeviceArray
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    stream = program()["stream"]
    terma = to_device(field_terma(shape, org, sp, case["gantry"],
                                  case["side"], seed), stream)
    box = DeviceArray((6,), np.int32)
    E.support_box(terma, shape, box, stream=stream)
    plan = program()["engine"].plan(
        shape, sp, cone_set(case["n_phi"], "physics",
                            source_of(case["gantry"])))
    dose = DeviceArray(shape)
    return State(kind="physics", E=E, plan=plan, terma=terma,
                 rho=to_device(densities_of(shape, seed), stream), dose=dose,
                 box=box, stream=stream, out=view(dose))


def run_physics(s):
    s["E"].convolve_rad(s["plan"], s["terma"], s["rho"], s["dose"], s["box"],
                        stream=s["stream"])
    return s["out"]


def prepare_gather(case, seed):
    from conehead_amd import engine as E
    from conehead_amd.device import DeviceArray
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    stream = program()["stream"]
    terma = to_device(field_terma(shape, org, sp, case["gantry"],
                                  case["side"], seed), stream)
    dose = DeviceArray(shape)
    return State(kind="gather", E=E, shape=shape, terma=terma, dose=dose,
                 box=DeviceArray((6,), np.int32), stream=stream,
                 plan=program()["engine"].plan(shape, sp,
                                               cone_set(case["n_phi"])),
                 out=view(dose))


def run_gather(s):
    E = s["E"]
    E.support_box(s["terma"], s["shape"], s["box"], stream=s["stream"])
    E.convolve(s["plan"], s["terma"], s["dose"], s["box"],
               stream=s["stream"])
    return s["out"]


def density_grids(case):
    src = shape_of(case)
    dst = (case["n"], case["n"], case["nz"])
    return (src,) + grid_of(src, case["mm"]) + (dst,) + \
        grid_of(dst, case["dose_mm"])


def prepare_density(case, seed):
    from conehead_amd.device import DeviceArray
    src, _, _, dst, _, _ = grids = density_grids(case)
    ct, labels = ct_of(src, seed)
    stream = program()["stream"]
    rho, out = DeviceArray(src), DeviceArray(dst)
    return State(kind="density", grids=grids, ct=to_device(ct, stream),
                 labels=to_device(labels, stream), rho=rho, dst=out,
                 stream=stream, out={"ct": view(rho), "dose": view(out)})


def run_density(s):
    from conehead_amd.density import ct_to_density, resample
    ct_to_density(s["ct"], CT_CURVE, s["labels"], CT_OVERRIDES, s["rho"],
                  stream=s["stream"])
    resample(s["rho"], *s["grids"], d_dst=s["dst"], stream=s["stream"])
    return s["out"]


# ------------------------------------------------------------------- work --

def work(case):
    kind = case["kind"]
    if kind == "batch":
        return total(beam_work(shape, mm, side) for shape, mm, _, beams
                     in requests_of(case) for _, side in beams)
    if kind == "density":
        src, _, _, dst, _, _ = density_grids(case)
        n, m = math.prod(src), math.prod(dst)
        return {"bytes": 7 * n + 36 * m, "flops": 4 * n + 40 * m}
    shape = shape_of(case)
    n = math.prod(shape)
    if kind == "replay":
        return total([beam_work(shape, case["mm"], 10.0)] * case["beams"])
    if kind in ("beam", "calculate"):
        return beam_work(shape, case["mm"], case["side"] or 10.0)
    path = sum(shape) / 3.0
    lit = lit_share(shape, case["mm"], case["side"])
    if kind == "physics":
        # every voxel's path to the field along the cones that reach it
        taps = n * 12 * case["n_phi"] * path * lit
        return {"bytes": 12 * n, "flops": 12 * taps}
    if kind == "gather":
        return {"bytes": 8 * n,
                "flops": 2 * n * 12 * case["n_phi"] * path * lit}
    return {"bytes": 24 * n, "flops": fft_flops(shape)}


def total(works):
    works = list(works)
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def lit_share(shape, mm, side):
    wide = (math.prod(shape) ** (1.0 / 3)) * mm / 10.0
    return min(1.0, (side / wide) ** 2)


def fft_flops(shape):
    f = math.prod(2 * n - 1 for n in shape)
    return 5.0 * f * math.log2(f) + 3.0 * f


def beam_work(shape, mm, side):
    """Densities read, TERMA written and read, dose written; the walk of
    the lit voxels, the spectrum sum and the transforms."""
    n = math.prod(shape)
    walk = n * lit_share(shape, mm, side) * (sum(shape) / 3.0 * 8 + 200)
    return {"bytes": 16 * n, "flops": walk + fft_flops(shape)}


# ------------------------------------------- the same in 64 bits, plainly --

def geometry(gantry):
    """Source position, beam direction and world -> source rotation."""
    phi = (90 - float(gantry)) % 360
    pos = np.array([100.0 * np.cos(phi * np.pi / 180),
                    100.0 * -np.sin(phi * np.pi / 180), 0.0])
    g = float(gantry) * np.pi / 180
    rot = np.array([[np.cos(g), -np.sin(g), 0], [np.sin(g), np.cos(g), 0],
                    [0, 0, 1.0]])
    axes = [rot @ np.eye(3)[k] for k in range(3)]
    return pos, axes[1], np.linalg.inv(np.array(axes).T)


def leaf_area(rows, cols):
    a = np.ones((rows, cols), np.float32)
    for k, v in enumerate((0.20, 0.50, 0.75)):
        a[k] = v
    for k, v in enumerate((0.20, 0.50, 0.75)):
        a[rows - 1 - k] = v
    a[:, -15:] *= np.linspace(1.0, 0.0, 15)
    return 1 - a


def raster_of(aperture):
    """Transmission at 0.1 mm over 40 x 40 cm of the isocentre plane."""
    if aperture[0] == "square":
        r = np.zeros((4000, 4000), np.float32)
        lo, hi = (int(2000 + s * aperture[1] / 2 * 100) for s in (-1, 1))
        r[lo:hi, lo:hi] = 1
        return r
    bound, a, b, jx, jy = [np.floor(np.asarray(v) * 10).astype(int)
                           for v in aperture[1:]]
    width = bound[-1] - bound[0]
    bank = np.ones((width, 4000), np.float32)
    for k in range(len(a)):
        r0, r1 = bound[k] - bound[0], bound[k + 1] - bound[0]
        bank[r0:r1, :2000 + a[k]] = leaf_area(r1 - r0, 2000 + a[k])
    for k in range(len(b)):
        r0, r1 = bound[k] - bound[0], bound[k + 1] - bound[0]
        bank[r0:r1, 2000 + b[k]:3999] = leaf_area(
            r1 - r0, 1999 - b[k])[::-1, ::-1]
    bank[:, :2000 + jx[0]] = 0
    bank[:, 2000 + jx[1]:] = 0
    bank[:max(0, width // 2 + jy[0])] = 0
    bank[max(0, width // 2 + jy[1]):] = 0
    r = np.zeros((4000, 4000), np.float32)
    r[2000 - width // 2:2000 - width // 2 + width] = bank
    return r


def dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def terma64(rho, org, sp, gantry, aperture):
    """TERMA of one beam: 27 sub-samples per voxel through the aperture,
    the voxel walk toward the source, the three sources and the spectrum."""
    S = SETTINGS
    pos, vy, tr = geometry(gantry)
    src = [float(v) for v in pos]
    vy = [float(v) for v in vy]
    tr = tr.tolist()
    shape = tuple(rho.shape)
    rho = rho.double().contiguous()
    dev = rho.device
    raster = torch.from_numpy(raster_of(aperture)).to(dev)
    c = [torch.arange(shape[a], dtype=torch.float64, device=dev)
         .mul(sp[a]).add(org[a]).reshape([-1 if a == b else 1
                                          for b in range(3)])
         for a in range(3)]
    nsrc = dot(vy, src)

    def on_plane(u):
        si = -nsrc / dot(vy, u)
        pp = [src[a] + si * u[a] for a in range(3)]
        return dot(tr[0], pp), dot(tr[2], pp)

    blocked = torch.zeros(shape, dtype=torch.float64, device=dev)
    ns = S["fluenceResampling"]
    off = [float(v) / ns for v in sp]
    for k in itertools.product(range(ns), repeat=3):
        u = [src[a] - (c[a] - sp[a] / 2 + off[a] / 2 + off[a] * k[a])
             for a in range(3)]
        q0, q2 = on_plane(u)
        i = torch.floor(q0 * 100.0) + 2000.0
        j = torch.floor(q2 * 100.0) + 2000.0
        ok = (i >= 0) & (i <= 3999) & (j >= 0) & (j <= 3999)
        i = (i.clamp(0, 3999).long() - 1) % 4000
        j = (j.clamp(0, 3999).long() - 1) % 4000
        v = torch.where(ok, raster[i, j].double(), torch.zeros_like(q0))
        blocked += v / float(ns ** 3)
    out = torch.zeros(shape, dtype=torch.float64, device=dev)
    at = torch.nonzero(blocked.reshape(-1)).reshape(-1)
    if not len(at):
        return out
    bl = blocked.reshape(-1)[at]
    cur = [at // (shape[1] * shape[2]), (at // shape[2]) % shape[1],
           at % shape[2]]
    r = [src[a] - c[a].reshape(-1)[cur[a]] for a in range(3)]
    mag = torch.sqrt(dot(r, r))
    d = [v / mag for v in r]
    step = [torch.where(v < 0, -1, 1) for v in d]
    dt = [torch.where(v == 0, torch.full_like(v, 1e9), sp[a] / v.abs())
          for a, v in enumerate(d)]
    t = [torch.where(v == 0, torch.full_like(v, 1e9),
                     (sp[a] / 2) / v.abs()) for a, v in enumerate(d)]
    flat = rho.reshape(-1)
    deff, last = torch.zeros_like(mag), torch.zeros_like(mag)
    while True:
        live = torch.ones_like(mag, dtype=torch.bool)
        for a in range(3):
            live &= (cur[a] >= 0) & (cur[a] < shape[a])
        if not bool(live.any()):
            break
        here = (cur[0] * shape[1] + cur[1]) * shape[2] + cur[2]
        m0 = (t[0] < t[1]) & (t[0] < t[2])
        m1 = ~(t[0] < t[1]) & (t[1] < t[2])
        ms = (m0, m1, ~(m0 | m1))
        now = torch.where(m0, t[0], torch.where(m1, t[1], t[2]))
        deff += torch.where(live, flat[torch.where(live, here, 0)] *
                            (now - last), torch.zeros_like(now))
        last = now
        for a in range(3):
            t[a] = torch.where(ms[a], t[a] + dt[a], t[a])
            cur[a] = torch.where(ms[a], cur[a] + step[a], cur[a])
    q0, q2 = on_plane(r)
    oad = torch.sqrt(q0 * q0 + q2 * q2)
    ra = oad * S["zAnn"] / 100.0
    fa = torch.where((ra >= S["rInner"]) & (ra <= S["rOuter"]),
                     S["sAnn"] * (100.0 - S["zAnn"]) ** 2 /
                     (mag - S["zAnn"]) ** 2, torch.zeros_like(ra))
    re = oad.clamp(min=2.0) * S["zExp"] / 100.0
    fe = S["sExp"] / re * torch.exp(-S["kExp"] * re) * \
        (100.0 - S["zExp"]) ** 2 / (mag - S["zExp"]) ** 2
    flu = (S["sPri"] * (100.0 / mag) ** 2 + fa + fe) * bl
    soft = torch.where(oad < S["softLimit"],
                       1.0 / (1.0 - S["softRatio"] * oad),
                       torch.ones_like(oad))
    acc = torch.zeros_like(mag)
    x, y = np.array(WATER, dtype=np.float32).astype(np.float64).T
    for e, w in S["energy_weights"].items():
        e, w = float(np.float32(e)), float(np.float32(w))
        mu = float(np.interp(e, x, y))
        acc += w * flu * torch.exp(-mu * soft * deff) * e * mu
    out.reshape(-1)[at] = acc * (1.0 + oad * S["hornRatio"]) * bl
    return out


def directions(n_phi, semantics, gantry=None):
    """Cone directions (12 azimuths, then the polar angles), their rows of
    the kernel table and the table."""
    phis, rows = cone_table(n_phi)
    pi = 3.14159265359 if semantics == "convolve_c" else math.pi
    frame = np.eye(3)
    if semantics == "physics":      # the cones turn with the beam
        g = float(gantry) * np.pi / 180
        rot = np.array([[np.cos(g), -np.sin(g), 0],
                        [np.sin(g), np.cos(g), 0], [0, 0, 1.0]])
        frame = [rot @ np.eye(3)[k] for k in range(3)]
    out = []
    for th in np.linspace(0, 360, 12, endpoint=False):
        for p in phis:
            a = float(th) * pi / 180.0
            b = float(p if semantics == "convolve_c" else 180.0 - p) * \
                pi / 180.0
            d = [math.cos(a) * math.sin(b), math.sin(a) * math.sin(b),
                 math.cos(b)]
            if semantics == "convolve_c":
                n = 1.0 / dot(d, d)
                d = [float(np.ceil(v * n * 100000)) * 0.00001 for v in d]
            else:                   # the polar axis is y
                d = [d[0], d[2], d[1]]
                n = math.sqrt(dot(d, d))
                d = [v / n for v in d]
                d = [sum(d[a] * frame[a][k] for a in range(3))
                     for k in range(3)]
            out.append(d)
    return np.array(out), np.tile(np.arange(n_phi), 12), rows


def walks(dirs, shape, sp):
    """Per step of every cone's walk from a voxel's centre: the offsets,
    the crossing value and whether the offset can lie in the grid."""
    n = len(dirs)
    step = np.where(dirs < 0, -1, 1)
    ad = np.abs(dirs)
    with np.errstate(divide="ignore"):
        t = np.where(ad == 0, 1e9, (sp / 2) / ad)
        dt = np.where(ad == 0, 1e9, sp / ad)
    cur = np.zeros((n, 3), np.int64)
    who = np.arange(n)
    while True:
        live = (np.abs(cur) < np.array(shape)).all(axis=1)
        if not live.any():
            return
        a = np.where(t[:, 0] < t[:, 1], np.where(t[:, 0] < t[:, 2], 0, 2),
                     np.where(t[:, 1] < t[:, 2], 1, 2))
        now = t[who, a]
        yield cur.copy(), now.copy(), live
        t[who, a] += dt[who, a]
        cur[who, a] += step[who, a]


def conv64(terma, sp, n_phi, semantics):
    """The cone convolution: every cone's increments summed into one kernel
    on a frame that holds the linear convolution."""
    shape = tuple(terma.shape)
    dirs, row, cum = directions(n_phi, semantics)
    off = 50.0 if semantics == "convolve_c" else 5.0
    frame = [smooth(2 * n - 1) for n in shape]
    K = np.zeros(frame)
    prev = np.zeros(len(dirs))
    done = np.zeros(len(dirs), bool)
    for cur, now, live in walks(dirs, shape, sp):
        idx = np.abs(np.floor(now * 100.0 - off))
        if semantics == "convolve_c":
            done |= idx > 5995
        idx = np.minimum(idx, 5995).astype(int)
        v = cum[row, idx]
        ok = live & ~done
        o = cur[ok]
        np.add.at(K, (o[:, 0], o[:, 1], o[:, 2]), v[ok] - prev[ok])
        prev = v
    dev = terma.device
    A = torch.fft.rfftn(terma.double(), s=frame)
    A *= torch.fft.rfftn(torch.from_numpy(K).to(dev))
    return torch.fft.irfftn(A, s=frame)[:shape[0], :shape[1], :shape[2]]


def smooth(n):
    while True:
        k = n
        for q in (2, 3, 5):
            while k % q == 0:
                k //= q
        if k == 1:
            return n
        n += 1


def rad64(terma, rho, sp, n_phi, gantry):
    """The convolution with the kernel looked up at the distance through
    the densities, from every receiving voxel back along every cone."""
    shape = tuple(terma.shape)
    dev = terma.device
    T, rho = terma.double(), rho.double()
    dirs, row, cum = directions(n_phi, "physics", gantry)
    steps = list(walks(dirs, shape, sp))
    dose = torch.zeros(shape, dtype=torch.float64, device=dev)
    for c in range(len(dirs)):
        tab = torch.from_numpy(cum[row[c]]).to(dev)
        R, prev = torch.zeros_like(dose), torch.zeros_like(dose)
        last = 0.0
        for cur, now, live in steps:
            if not live[c]:
                break
            o = cur[c]
            v = tuple(slice(max(0, o[a]), shape[a] + min(0, o[a]))
                      for a in range(3))
            s = tuple(slice(max(0, -o[a]), shape[a] - max(0, o[a]))
                      for a in range(3))
            R[v] += rho[s] * (now[c] - last)
            last = now[c]
            idx = torch.floor(R[v] * 100.0 - 5.0).abs().clamp(max=5995)
            val = tab[idx.long()]
            dose[v] += T[s] * (val - prev[v])
            prev[v] = val
    return dose


def ct64(ct, labels):
    x, y = np.array(CT_CURVE).T
    lut = torch.from_numpy(np.interp(np.arange(-32768, 32768), x, y)).cuda()
    rho = lut[torch.from_numpy(ct).cuda().long() + 32768]
    lab = torch.from_numpy(labels).cuda()
    for k, v in CT_OVERRIDES.items():
        rho[lab == k] = float(np.float32(v))
    return rho


def resample64(src, org, sp, dst, dorg, dsp):
    """Trilinear on linspace axes, 0 outside, the x and y axes of the
    result exchanged as the reference lays it out."""
    at = []
    for a in range(3):
        n = src.shape[a]
        nodes = np.linspace(org[a], org[a] + n * sp[a], n)
        p = np.linspace(dorg[a], dorg[a] + dst[a] * dsp[a], dst[a])
        i = np.clip(np.searchsorted(nodes, p) - 1, 0, n - 2)
        f = (p - nodes[i]) / (nodes[i + 1] - nodes[i])
        ok = (p >= nodes[0]) & (p <= nodes[-1])
        at.append([torch.from_numpy(v).cuda().reshape(
            [-1 if a == b else 1 for b in range(3)]) for v in (i, f, ok)])
    out = 0.0
    for e in itertools.product((0, 1), repeat=3):
        w = 1.0
        for a in range(3):
            w = w * (at[a][1] if e[a] else 1.0 - at[a][1])
        out = out + w * src[at[0][0] + e[0], at[1][0] + e[1],
                            at[2][0] + e[2]].double()
    ok = at[0][2] & at[1][2] & at[2][2]
    return torch.where(ok, out, torch.zeros_like(out)).transpose(0, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "density":
        src, org, sp, dst, dorg, dsp = density_grids(case)
        rho = ct64(*ct_of(src, seed))
        return {"ct": rho,
                "dose": resample64(rho, org, sp, dst, dorg, dsp)}
    if kind == "batch":
        got = []
        for i, (shape, mm, n_phi, beams) in enumerate(requests_of(case)):
            org, sp = grid_of(shape, mm)
            rho = torch.from_numpy(densities_of(shape, seed + 1000 * i))
            for g, side in beams:
                t = terma64(rho.cuda(), org, sp, g, ("square", side))
                got.append(conv64(t, sp, n_phi, "convolve_c"))
        return got
    shape = shape_of(case)
    org, sp = grid_of(shape, case["mm"])
    if kind == "dropin":
        t, dose, _ = dropin_inputs(case, seed)
        return torch.from_numpy(dose).cuda() + conv64(
            torch.from_numpy(t).cuda(), sp, case["n_phi"], "convolve_c")
    if kind == "gather":
        t = field_terma(shape, org, sp, case["gantry"], case["side"], seed)
        return conv64(t, sp, case["n_phi"], "convolve_c")
    if kind == "physics":
        t = field_terma(shape, org, sp, case["gantry"], case["side"], seed)
        return rad64(t, torch.from_numpy(densities_of(shape, seed)).cuda(),
                     sp, case["n_phi"], case["gantry"])
    if kind == "replay":
        rho = torch.from_numpy(densities_of(shape, seed)).cuda()
        return [conv64(terma64(rho, org, sp, g, ap), sp, case["n_phi"],
                       "convolve_c") for g, ap in replay_beams(case, seed)]
    semantics = case.get("semantics", "convolve_c")
    if kind == "beam":
        rho = torch.from_numpy(densities_of(shape, seed)).cuda()
        ap = aperture_of(case["side"], np.random.default_rng([seed, 5]))
    else:
        if case.get("ct"):
            cshape, corg, csp = ct_grid(case)
            rho = ct64(*ct_of(cshape, seed))
            rho = resample64(rho, corg, csp, shape, org, sp)
        else:
            # the reference's interpolation exchanges x and y
            rho = torch.from_numpy(densities_of(shape, seed)).cuda() \
                .transpose(0, 1)
        ap = ("square", case["side"])
    t = terma64(rho.float(), org, sp, case["gantry"], ap)
    return {"dose": conv64(t, sp, case["n_phi"], semantics), "terma": t}
