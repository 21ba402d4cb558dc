"""What is kept between calls, on the CPU: the drop-in's buffers, the way its
result reaches doses of any layout, the pools and the tuned tiles, with numpy
arrays standing in for device and pinned memory."""
import numpy as np
import pytest

from conehead_amd import _lib, batch, convolve_c, device


class Dev:
    """A DeviceArray's interface on host memory."""

    def __init__(self, shape, dtype=np.float32):
        self.a = np.zeros(shape, dtype)
        self.shape, self.dtype = self.a.shape, self.a.dtype
        self.nbytes, self.size = self.a.nbytes, self.a.size

    def upload(self, arr, stream=None):
        self.a[...] = arr
        return self

    def download(self, out=None, stream=None):
        out = np.empty_like(self.a) if out is None else out
        assert out.flags.c_contiguous and out.dtype == self.dtype
        out[...] = self.a
        return out


class Pinned:
    """A HostBuffer's; `made` counts the allocations."""
    made = 0
    fail = False

    def __init__(self, nbytes):
        if Pinned.fail:
            raise _lib.CHError(_lib.CH_ERR_NOMEM, "no pinned memory")
        Pinned.made += 1
        self.nbytes = nbytes
        self.mem = np.zeros(nbytes, np.uint8)
        self.ptr = self.mem.ctypes.data


class FakePlan:
    def spectrum(self):
        pass


@pytest.fixture
def dropin(monkeypatch):
    """convolve_c's host path with a convolution that doubles TERMA."""
    def doubled(plan, t, part):
        part.a[...] = 2 * t.a

    def doubled64(plan, t, dose, box):
        dose.a[...] += 2 * t.a

    monkeypatch.setattr(convolve_c, "DeviceArray", Dev)
    monkeypatch.setattr(convolve_c, "HostBuffer", Pinned)
    monkeypatch.setattr(convolve_c, "_convert",
                        lambda dst, src: dst.upload(src.a))
    monkeypatch.setattr(convolve_c._engine, "convolve_fft", doubled)
    monkeypatch.setattr(convolve_c._engine, "convolve_f64", doubled64)
    monkeypatch.setattr(convolve_c._engine, "support_box", lambda *a: None)
    monkeypatch.setattr(_lib, "lib", _lib.load)
    monkeypatch.setattr(convolve_c, "_BUFS", type(convolve_c._BUFS)())
    if hasattr(convolve_c, "_PINNED"):
        monkeypatch.setattr(convolve_c, "_PINNED", {})
    monkeypatch.setattr(Pinned, "made", 0)
    monkeypatch.setattr(Pinned, "fail", False)

    def call(shape, dose=None, fft=True):
        t = np.random.default_rng(sum(shape)).random(shape)
        dose = np.ones(shape) if dose is None else dose
        want = dose + 2 * t.astype(np.float32)
        convolve_c._run(FakePlan(), shape, t, dose, fft)
        assert np.array_equal(dose, want)
    return call


SHAPES = [(4, 5, n) for n in (11, 3, 7, 5, 9, 2)]


def test_dropin_pinned_target_serves_every_shape(dropin):
    """One pinned buffer as large as the largest result, not one per shape:
    a caller that goes round more shapes than are kept allocates none."""
    for _ in range(3):
        for shape in SHAPES:
            dropin(shape)
    assert Pinned.made == 1
    dropin((4, 5, 12))                     # a larger one replaces it
    assert Pinned.made == 2


def test_dropin_gather_takes_no_pinned_memory(dropin):
    for shape in SHAPES:
        dropin(shape, fft=False)
    assert Pinned.made == 0


def test_dropin_without_pinned_memory(dropin, monkeypatch):
    """Results past the kept size, or no pinned memory to be had: ordinary
    memory takes its place."""
    monkeypatch.setattr(Pinned, "fail", True)
    dropin((4, 5, 6))
    monkeypatch.setattr(Pinned, "fail", False)
    monkeypatch.setattr(convolve_c, "_MAX_PINNED", 4 * 4 * 5 * 6 - 1)
    dropin((4, 5, 6))
    assert Pinned.made == 0


def test_dropin_drops_the_oldest_shape(dropin):
    for shape in SHAPES[:5]:
        dropin(shape)
    dropin(SHAPES[0])
    dropin(SHAPES[5])
    assert set(convolve_c._BUFS) == set(SHAPES) - {SHAPES[1]}


@pytest.mark.parametrize("layout", ["C", "F", "swapped", "step", "slice",
                                    "reversed", "unaligned"])
def test_dropin_dose_layouts(dropin, layout):
    shape = (6, 5, 7)
    dose = {"C": lambda: np.ones(shape),
            "F": lambda: np.ones(shape, order="F"),
            "swapped": lambda: np.ones((5, 6, 7)).transpose(1, 0, 2),
            "step": lambda: np.ones((6, 5, 14))[:, :, ::2],
            "slice": lambda: np.ones((6, 9, 7))[:, 2:7],
            "reversed": lambda: np.ones(shape)[::-1, :, ::-1],
            "unaligned": lambda: np.frombuffer(
                bytearray(1) + bytearray(np.ones(shape).tobytes()), np.uint8)
            [1:].view(np.float64).reshape(shape)}[layout]()
    dropin(shape, dose)


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 1, 0), (1, 0, 2),
                                   (0, 2, 1), (1, 2, 0), (2, 0, 1)])
@pytest.mark.parametrize("shape", [(6, 5, 7), (8, 16, 16), (1, 17, 9),
                                   (33, 1, 40), (70, 65, 130)])
def test_sum_into_any_axis_order(monkeypatch, order, shape):
    """Tiles and remainders, one and four threads, axes reversed and of
    every other element: numpy's sum, and nothing beside the dose's own
    elements."""
    monkeypatch.setattr(_lib, "lib", _lib.load)
    rng = np.random.default_rng(sum(shape))
    part = rng.random(shape).astype(np.float32)
    for step in (slice(None), slice(None, None, -1), slice(None, None, 2)):
        n = 2 if step.step == 2 else 1
        whole = rng.random([n * shape[a] for a in order])
        before = whole.copy()
        view = [a.transpose(np.argsort(order))[step, step, step]
                for a in (whole, before)]
        assert view[0].shape == shape
        convolve_c._add(view[0], part)
        view[1] += part
        assert np.array_equal(whole, before)


def test_sum_into_overlapping_elements(monkeypatch):
    """Doses whose elements share memory stay numpy's."""
    monkeypatch.setattr(_lib, "lib", _lib.load)
    part = np.ones((4, 5, 6), np.float32)
    for strides in ((8, 8, 8), (8, 0, 16), (16, 8, 40), (8, 16, 8)):
        base = np.zeros(400)
        want = base.copy()
        dose, ref = [np.lib.stride_tricks.as_strided(b, (4, 5, 6), strides)
                     for b in (base, want)]
        convolve_c._add(dose, part)
        np.add(ref, part, out=ref)
        assert np.array_equal(base, want)


class Block:
    """A pooled buffer of either kind; `live` holds those not freed."""
    live = []
    ptr = 1

    def __init__(self, shape, dtype=np.uint8):
        self.shape = shape if isinstance(shape, tuple) else (shape,)
        self.dtype = np.dtype(dtype)
        self.nbytes = int(np.prod(self.shape)) * self.dtype.itemsize
        Block.live.append(self)

    def free(self):
        Block.live.remove(self)
        self.ptr = None


@pytest.fixture(params=["device", "host"])
def pool(request, monkeypatch):
    """(pool of at most 100 idle bytes, its buffer of n bytes)"""
    monkeypatch.setattr(Block, "live", [])
    if request.param == "device":
        monkeypatch.setattr(batch, "DeviceArray", Block)
        p = batch.DevicePool(max_free_bytes=100)
        return p, lambda n: p.get((n,), np.uint8)
    monkeypatch.setattr(device, "HostBuffer", Block)
    p = device.HostPool(max_free_bytes=100)
    return p, p.get


def test_full_pool_keeps_the_shape_in_use(pool):
    """Buffers of shapes that are gone make room: a pool filled by earlier
    shapes keeps the present one's."""
    p, get = pool
    old = [get(n) for n in (30, 31, 32)]
    for b in old:
        p.put(b)
    a, b = get(40), get(40)
    p.put(a)                               # the two oldest go
    p.put(b)
    assert Block.live == [a, b] and p._bytes == 80
    assert {get(40), get(40)} == {a, b} and p._bytes == 0
    c = get(101)                           # larger than the pool
    for x in (a, c, b):
        p.put(x)
    assert Block.live == [a, b]
    p.put(get(19))                         # fits beside them
    assert get(40) is b                    # the size is in use again
    p.put(b)
    p.put(get(20))                         # so the 19 bytes go
    assert sorted(x.nbytes for x in Block.live) == [20, 40, 40]
    p.clear()
    assert Block.live == [] and p._bytes == 0 and not p._free


def test_pinned_bytes_are_bounded(monkeypatch):
    """try_get counts what is handed out: buffers that callers keep end the
    pinned memory of a pool, idle ones of other sizes make room, and what is
    dropped can be had again."""
    monkeypatch.setattr(Block, "live", [])
    monkeypatch.setattr(device, "HostBuffer", Block)
    p = device.HostPool(max_free_bytes=60, max_bytes=100)
    kept = [p.try_get(40), p.try_get(40)]
    assert None not in kept and p.try_get(40) is None
    p.put(kept.pop())
    assert p.try_get(60) is not None         # the idle 40 bytes are freed
    assert sorted(b.nbytes for b in Block.live) == [40, 60]
    assert p.try_get(1) is None
    p.put(kept.pop())
    idle = p.try_get(40)
    assert idle is not None and p.try_get(40) is None

    def none(nbytes):
        raise _lib.CHError(_lib.CH_ERR_NOMEM, "no pinned memory")

    monkeypatch.setattr(device, "HostBuffer", none)
    p.put(idle)
    assert p.try_get(30) is None and p.try_get(40) is None


def test_short_memory_empties_the_pools(monkeypatch):
    """An allocation that fails for want of memory is tried again without
    the idle buffers of every pool, and fails when none are left."""
    class Lib:
        room = 100

        def ch_malloc(self, p, nbytes):
            if nbytes > Lib.room:
                return _lib.CH_ERR_NOMEM
            Lib.room -= nbytes
            p._obj.value = 1 + nbytes
            return _lib.CH_OK

        def ch_free(self, ptr):
            Lib.room += ptr - 1
            return _lib.CH_OK

        ch_host_alloc, ch_host_free = ch_malloc, ch_free

    one = Lib()
    monkeypatch.setattr(_lib, "lib", lambda: one)
    monkeypatch.setattr(device, "_POOLS", type(device._POOLS)())
    pools = batch.DevicePool(), device.HostPool()
    a, h = pools[0].get((40,), np.uint8), pools[1].get(30)
    pools[0].put(a)
    pools[1].put(h)
    assert Lib.room == 30
    b = device.DeviceArray((80,), np.uint8)
    assert Lib.room == 20 and pools[0]._bytes == pools[1]._bytes == 0
    with pytest.raises(_lib.CHError) as e:
        device.HostBuffer(21)
    assert e.value.status == _lib.CH_ERR_NOMEM
    b.free()
    assert Lib.room == 100
    monkeypatch.undo()       # the freed buffers above end on the fake library


def test_tiles_of_earlier_workgroups_are_not_read(tmp_path, monkeypatch):
    """Tiles timed when the gather's workgroups were others stay in the cache
    file; tuning times anew."""
    import json
    from types import SimpleNamespace
    from conehead_amd import autotune

    class Timed(Exception):
        pass

    def timing(*a):
        raise Timed

    path = tmp_path / "tiles.json"
    path.write_text(json.dumps({"10x11x12/6": {
        "tile": [1, 1, 64], "ms": {"1x1x64": 1.0}}}))
    monkeypatch.setattr(autotune, "CACHE_PATH", str(path))
    monkeypatch.setattr(autotune, "_memo", {})
    monkeypatch.setattr(autotune, "Stream", timing)
    plan = SimpleNamespace(shape=(10, 11, 12), n_cones=6,
                           set_tile=lambda *t: None)
    with pytest.raises(Timed):
        autotune.tune(plan)


def test_unused_instances_can_be_copied():
    """A Conehead that has not computed holds nothing of the process."""
    import copy
    import pickle
    from conehead_amd.conehead import Conehead
    for one in (copy.deepcopy(Conehead()),
                pickle.loads(pickle.dumps(Conehead()))):
        assert one.dose_grid is None
